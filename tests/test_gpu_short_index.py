"""Batch plans over streams whose index was kept from a library that wrote
shorter ones: a plan launched again reads the bytes that are there by then."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402
from tests.golden import gen  # noqa: E402

pytestmark = pytest.mark.gpu

L, EB = 36, 1e-3


@pytest.fixture(scope="module")
def zccl():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from zccl_amd import batch, codec

    torch.cuda.set_device(0)
    return codec, batch


def stored(codec, cx, n, T):
    """The stream with an index as it was before the carries."""
    data = torch.zeros(codec.worst_case_bytes(n, L, T), dtype=torch.uint8, device="cuda")
    data[: cx.size] = torch.from_numpy(np.ascontiguousarray(cx)).cuda()
    s = codec.from_bytes(data, n, L, T)
    return codec.DeviceStream(data, s.index[: s.size_offset + 32].clone(), n, L, T)


@pytest.mark.parametrize("n,T", [(2_311, 1), (100_003, 4)])
def test_plans_follow_the_bytes(zccl, n, T):
    codec, batch = zccl
    print("[gpu] short index plans", n, T, flush=True)
    cs = [O.compress(gen.make("grf", n, 60 + i), EB, L, T) for i in range(3)]
    s, full = stored(codec, cs[0], n, T), codec.upload(cs[2], n, L, T)
    y, out = torch.empty(n, device="cuda"), codec.empty_stream(n, L, T)
    dec, add = batch.decompress_plan([s], [EB], [y]), batch.homsum_plan([[s, full]], [out])
    for c in (cs[0], cs[1]):
        new = stored(codec, c, n, T)
        s.data.copy_(new.data)
        s.index.copy_(new.index)
        ws = codec.Workspace(max(dec.tiles, add.tiles))
        dec.launch(ws)
        add.launch(ws)
        codec.check_errors(ws)
        assert np.array_equal(y.cpu().numpy().view(np.uint32), O.decompress(c, n, EB, L, T).view(np.uint32))
        assert np.array_equal(out.to_host(), O.homsum([c, cs[2]], n, L, T))
