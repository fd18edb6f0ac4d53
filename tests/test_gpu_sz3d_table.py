"""3-D streams of many sub-volumes: the table of one lane per sub-volume at 63,
64, 65 and more of them, of different sizes, for each block side's kernels.
Stream bytes and values equal the oracle's."""
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


@pytest.mark.parametrize("dims,Bs,T", [
    ((67, 21, 35), 4, 63), ((67, 21, 35), 4, 64), ((67, 21, 35), 8, 65), ((131, 9, 10), 3, 127), ((45, 38, 37), 4, 128),
    ((45, 38, 37), 8, 200)])
def test_many_sub_volumes(sz, dims, Bs, T):
    print("[3d table]", dims, Bs, T, flush=True)
    x = gen.smooth3d(dims, T) * np.float32(20)
    c = O.compress3d(x, dims, Bs, 1e-3, T)
    s = sz.compress(torch.from_numpy(x).cuda(), Bs, 1e-3, T)
    assert np.array_equal(s.to_host(), c)
    y = sz.decompress(sz.upload(c, dims, Bs, 1e-3, T)).cpu().numpy().reshape(-1)
    assert np.array_equal(y.view(np.uint32), O.decompress3d(c, dims, Bs, 1e-3, T).view(np.uint32))
