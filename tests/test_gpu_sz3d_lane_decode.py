"""3-D decompress with block side 4 by lanes: rows of 32 to 256 blocks along z
(one, two and four waves of 64), segments of 8 blocks along x, far edges in every
direction, widths up to 32 with and without payloads wider than a wave's buffer,
sub-volumes of different sizes.  Bits equal the oracle's."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
from oracle import oracle as O  # noqa: E402
from tests.golden import gen  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sz():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from zccl_amd import sz3d

    return sz3d


@pytest.mark.parametrize("dims,T,amp", [
    ((4, 4, 128), 1, 20.0), ((1, 1, 125), 1, 20.0), ((5, 6, 253), 1, 20.0), ((32, 8, 256), 1, 20.0),
    ((33, 7, 257), 1, 20.0), ((70, 9, 300), 1, 20.0), ((37, 13, 515), 1, 20.0), ((9, 5, 1021), 1, 20.0),
    ((10, 6, 1024), 1, 20.0), ((67, 66, 290), 8, 20.0), ((75, 31, 190), 6, 20.0), ((41, 10, 140), 1, 3e4), ((5, 6, 124), 1, 20.0),
    ((41, 11, 331), 2, 1e6), ((6, 5, 1028), 1, 20.0), ((129, 40, 517), 2, 20.0)])
def test_values_equal_oracle(sz, dims, T, amp):
    print("[lane3d decode]", dims, T, amp, flush=True)
    x = gen.smooth3d(dims, T) * np.float32(amp)
    if amp > 100:  # payloads wider than a wave's buffer
        x = x + np.random.default_rng(T).normal(0, amp, dims).astype(np.float32)
        x[1, 1, 1] = 3e9
    c = O.compress3d(x, dims, 4, 1e-3, T)
    y = sz.decompress(sz.upload(c, dims, 4, 1e-3, T)).cpu().numpy().reshape(-1)
    assert np.array_equal(y.view(np.uint32), O.decompress3d(c, dims, 4, 1e-3, T).view(np.uint32))


def test_cut_stream_is_refused(sz):
    """A stream cut in its payloads or its widths, and a width byte above 32,
    raise the errors they did."""
    dims, T = (20, 12, 100), 2
    c = O.compress3d(gen.smooth3d(dims, 3) * np.float32(20), dims, 4, 1e-3, T)
    bad = c.copy()
    bad[8 * T + 3] = 77
    w = torch.zeros(sz.sizes(dims, 4, T)[1], dtype=torch.uint8, device="cuda")
    for b in (c[: c.size - 200], c[: 8 * T + 40], bad):
        sz.decompress(sz.upload(b, dims, 4, 1e-3, T), ws=w)
        with pytest.raises(Exception):
            sz.check(w)
    sz.decompress(sz.upload(c, dims, 4, 1e-3, T), ws=w)
    assert sz.check(w) == c.size
