"""Decompress under an index that holds no stream (size 0, as a failed parse
leaves it) is reported, also where no segment has a block: segments of one value
have nothing but their seed."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

L = 36


@pytest.mark.parametrize("n,T", [(1, 1), (4, 4), (5, 4), (37, 1), (300, 7)])
def test_no_stream(n, T):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from zccl_amd import batch, codec

    print("[gpu] empty index", n, T, flush=True)
    data = torch.zeros(codec.worst_case_bytes(n, L, T), dtype=torch.uint8, device="cuda")
    s = codec.DeviceStream(data, torch.zeros(codec.index_bytes(n, L, T), dtype=torch.uint8, device="cuda"), n, L, T)
    ws = codec.Workspace(codec.num_tiles(n, L, T))
    codec.decompress(s, 1e-3, ws=ws)
    assert ws.errors() == 16
    plan = batch.decompress_plan([s], [1e-3], [torch.empty(n, device="cuda")])
    plan.launch(ws)
    assert ws.errors() == 16
