"""Damaged 3-D streams, block side 4, at volumes that the lane decoder takes (one
wave to a row; three waves, far edges and kept planes): cut in the payloads, in a
sub-volume's widths and in the header's reach, a width above 32, sub-volume
offsets past the stream.  Each is reported, and the workspace serves the whole
stream afterwards."""
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


@pytest.mark.parametrize("dims,T,amp", [((256, 192, 256), 16, 20.0), ((131, 195, 515), 2, 20.0), ((66, 256, 1024), 1, 1e6)])
def test_damage_is_reported(sz, dims, T, amp):
    x = gen.smooth3d(dims, 3) * np.float32(amp)
    if amp > 100:  # payloads wider than a wave's buffer
        x = x + np.random.default_rng(T).normal(0, amp, dims).astype(np.float32)
    c = O.compress3d(x, dims, 4, 1e-3, T)
    last = 8 * T + int(c[8 * (T - 1): 8 * T].view(np.uint64)[0])  # the last sub-volume's first width

    def changed(at, value):
        b = c.copy()
        b[at: at + len(value)] = value
        return b

    def u64(v):
        return np.array([v], dtype=np.uint64).view(np.uint8)

    cases = {"payload cut": c[: c.size - 200], "the last byte gone": c[: c.size - 1], "half the stream": c[: c.size // 2],
             "widths cut": c[: last + 100], "only the header": c[: 8 * T + 1], "a width of 77": changed(8 * T + 3, [77]),
             "a width of 33": changed(last + 50, [33]), "an offset past the end": changed(8 * (T - 1), u64(c.size)),
             "an offset of 2^63": changed(8 * (T - 1), u64(1 << 63))}
    w = torch.zeros(sz.sizes(dims, 4, T)[1], dtype=torch.uint8, device="cuda")
    for name, b in cases.items():
        print("[lane3d damaged]", dims, T, name, flush=True)
        sz.decompress(sz.upload(np.ascontiguousarray(b), dims, 4, 1e-3, T), ws=w)
        with pytest.raises(Exception):
            sz.check(w)
    y = sz.decompress(sz.upload(c, dims, 4, 1e-3, T), ws=w)
    assert sz.check(w) == c.size
    assert np.array_equal(y.cpu().numpy().reshape(-1).view(np.uint32), O.decompress3d(c, dims, 4, 1e-3, T).view(np.uint32))
