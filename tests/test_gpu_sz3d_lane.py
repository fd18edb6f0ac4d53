"""3-D compress with block side 4: one lane per block, runs of 63 blocks to a
wave, tiles of 4 or 12 waves.  Stream bytes equal the oracle's."""
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


# A run, a tile and one more block along z; sides of 1 and 3; sub-volumes that
# begin within a run; the tiles of 12 waves with ragged ends.
@pytest.mark.parametrize("dims,T,amp", [
    ((1, 1, 1), 1, 1.0), ((4, 4, 252), 1, 20.0), ((4, 4, 253), 1, 20.0), ((4, 4, 256), 1, 20.0),
    ((3, 5, 1009), 1, 20.0), ((1, 3, 1022), 1, 20.0), ((7, 61, 66), 5, 20.0), ((16, 16, 67), 8, 20.0),
    ((9, 33, 70), 3, 1e4), ((13, 30, 65), 4, 1e6), ((233, 239, 241), 7, 50.0), ((240, 240, 240), 1, 1e6)])
def test_stream_equals_oracle(sz, dims, T, amp):
    print("[lane3d]", dims, T, amp, flush=True)
    x = gen.smooth3d(dims, T) * np.float32(amp)
    if amp > 100:  # payloads wider than a wave's buffer
        x = x + np.random.default_rng(T).normal(0, amp, dims).astype(np.float32)
    s = sz.compress(torch.from_numpy(x).cuda(), 4, 1e-3, T)
    assert np.array_equal(s.to_host(), O.compress3d(x, dims, 4, 1e-3, T))
