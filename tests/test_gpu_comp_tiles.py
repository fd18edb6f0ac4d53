"""Lane compress, one or two tiles to a workgroup: totals of 256 tiles (one
each), 257 (a pair short of its second) and 258, of one stream, of equal ones
launched together and of mixed ones.  Against the oracle, byte for byte."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu

L, TILE = 36, 256 * 36


def sizes(tiles, k):
    """k sizes of together `tiles` tiles (a last tile of 5 values each)."""
    per = [tiles // k + (1 if i < tiles % k else 0) for i in range(k)]
    return [(p - 1) * TILE + 6 for p in per]


@pytest.mark.parametrize("tiles,k", [(256, 1), (257, 1), (258, 1), (256, 2), (258, 2), (270, 6), (256, 3), (257, 3), (259, 5)])
def test_tiles_of_a_workgroup(tiles, k):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from zccl_amd import batch, codec

    print("[gpu] comp tiles", tiles, k, flush=True)
    rng = np.random.default_rng(tiles * k)
    xs = [np.cumsum(rng.normal(0, 1, n)).astype(np.float32) for n in sizes(tiles, k)]
    ds = [torch.from_numpy(x).cuda() for x in xs]
    if k == 1:
        got = [codec.compress(ds[0], 1e-2, L, 1)]
    else:
        got = [codec.empty_stream(x.size, L, 1) for x in xs]
        batch.compress_plan(ds, [1e-2] * k, got).launch()
    torch.cuda.synchronize()
    codec.check_errors()
    for x, s in zip(xs, got):
        assert np.array_equal(s.to_host(), O.compress(x, 1e-2, L, 1))


@pytest.mark.parametrize("tiles", [(4096,), (4097,), (4103,), (4000, 97, 3)])
def test_sums_of_many_tiles(tiles):
    """Sums on both sides of the line at 4096 tiles of 64 blocks, alone and as
    a mixed batch, the last workgroup short of waves."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from zccl_amd import batch, codec

    print("[gpu] sum tiles", tiles, flush=True)
    rng = np.random.default_rng(sum(tiles))
    hs, ds, outs = [], [], []
    for t in tiles:
        n = t * 64 * L - 30
        xs = [np.cumsum(rng.normal(0, 1, n)).astype(np.float32) for _ in range(2)]
        hs.append([O.compress(x, 1e-2, L, 1) for x in xs])
        ds.append([codec.compress(torch.from_numpy(x).cuda(), 1e-2, L, 1) for x in xs])
        outs.append(codec.empty_stream(n, L, 1))
    if len(tiles) == 1:
        codec.homsum(ds[0], outs[0], stage=False)
    else:
        batch.homsum_plan(ds, outs).launch()
    torch.cuda.synchronize()
    codec.check_errors()
    for t, h, o in zip(tiles, hs, outs):
        assert np.array_equal(o.to_host(), O.homsum(h, t * 64 * L - 30, L, 1))
