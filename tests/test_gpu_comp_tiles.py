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
