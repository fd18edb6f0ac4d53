"""3-D compress with block side 4 at rows of 2^27 values and more.  Stream bytes
equal the oracle's for one row, whose blocks are of four values; several rows
are read back."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
from oracle import oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sz():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from zccl_amd import sz3d

    return sz3d


def row(n):
    part = np.cumsum(np.random.default_rng(4).normal(0, 0.02, 1 << 20)).astype(np.float32)
    return np.resize(part, n)


def test_one_long_row(sz):
    dims = (1, 1, (1 << 27) + 5)
    print("[long rows]", dims, flush=True)
    x = row(dims[2]).reshape(dims)
    s = sz.compress(torch.from_numpy(x).cuda(), 4, 1e-2, 1)
    assert np.array_equal(s.to_host(), O.compress3d(x, dims, 4, 1e-2, 1))


def test_long_rows_in_sub_volumes(sz):
    dims, T, eb = (2, 2, 1 << 27), 4, 1e-2
    print("[long rows]", dims, T, flush=True)
    x = torch.from_numpy(row(dims[2])).cuda() + torch.arange(4, device="cuda").reshape(2, 2, 1)
    s = sz.compress(x, 4, eb, T)
    y = sz.decompress(s)
    assert float((y.reshape(dims) - x).abs().max()) <= eb * 1.01
