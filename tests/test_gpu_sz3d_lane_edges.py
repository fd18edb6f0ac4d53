"""3-D compress with block side 4: far-edge blocks of every extent in every
direction (whole, 1, 2 and 3 values), in volumes of one block and of several,
in one sub-volume and in several of different sizes.  Stream bytes equal the
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


@pytest.mark.parametrize("ey", [1, 2, 3, 4])
@pytest.mark.parametrize("ez", [1, 2, 3, 4])
def test_far_edges(sz, ey, ez):
    print("[lane3d edges]", ey, ez, flush=True)
    for ex in (1, 2, 3, 4):
        for dims, T in (((ex, ey, ez), 1), ((4 + ex, 8 + ey, 60 + ez), 1), ((10 + ex, 6 + ey, 21 + ez), 6)):
            x = gen.smooth3d(dims, ex) * np.float32(50)
            x = x + np.random.default_rng(ex).normal(0, 20, dims).astype(np.float32)
            s = sz.compress(torch.from_numpy(x).cuda(), 4, 1e-3, T)
            assert np.array_equal(s.to_host(), O.compress3d(x, dims, 4, 1e-3, T)), (dims, T)
