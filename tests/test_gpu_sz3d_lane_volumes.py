"""3-D decompress with block side 4 at volumes large enough for the lane decoder
(three decode waves and one y-pass wave for each compute unit): rows of one, two,
three and four waves of 64 blocks, whole blocks and far edges in every
direction, sub-volumes of different sizes, widths up to 32.  Bits equal the
oracle's."""
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


def volume(dims, T, amp):
    x = gen.smooth3d(dims, T) * np.float32(amp)
    if amp > 100:  # payloads wider than a wave's buffer
        x = x + np.random.default_rng(T).normal(0, amp, dims).astype(np.float32)
        x[1, 1, 1] = 3e9
    return x


@pytest.mark.parametrize("dims,T,amp", [
    ((256, 192, 256), 16, 20.0), ((250, 190, 250), 16, 20.0), ((200, 350, 250), 9, 1e6),
    ((260, 192, 260), 4, 20.0), ((131, 195, 515), 2, 20.0), ((67, 257, 1021), 1, 20.0), ((66, 256, 1024), 1, 1e6)])
def test_values_equal_oracle(sz, dims, T, amp):
    print("[lane3d volumes]", dims, T, amp, flush=True)
    c = O.compress3d(volume(dims, T, amp), dims, 4, 1e-3, T)
    y = sz.decompress(sz.upload(c, dims, 4, 1e-3, T)).cpu().numpy().reshape(-1)
    assert np.array_equal(y.view(np.uint32), O.decompress3d(c, dims, 4, 1e-3, T).view(np.uint32))
