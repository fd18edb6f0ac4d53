"""Streams whose index was kept from a library that wrote shorter ones, as
outputs: what is handed to the kernels always has room for this library's index.
The library's device entry points are recorded here, not run."""
import ctypes
from types import SimpleNamespace

import pytest

torch = pytest.importorskip("torch")

from zccl_amd import batch, codec  # noqa: E402

N, L, T, EB = 10_007, 36, 4, 1e-3
WS = SimpleNamespace(max_tiles=1 << 16, nbytes=1 << 21, ptr=ctypes.c_void_p(4096), buf=None)


class OnDevice(torch.Tensor):
    """A host tensor that passes the device checks of the host layer."""

    is_cuda = True


def device(t):
    return t.as_subclass(OnDevice)


class Recorder:
    """The library, with its entry points that launch kernels recorded."""

    LAUNCH = ("zccl_compress_dev", "zccl_homsum_dev", "zccl_batch_compress_plan", "zccl_batch_homsum_plan",
              "zccl_decompress_dev", "zccl_parse_dev")

    def __init__(self, real):
        self.real, self.calls = real, []

    def __getattr__(self, name):
        if name not in self.LAUNCH:
            return getattr(self.real, name)

        def call(*a):
            self.calls.append((name, a))
            return 0
        return call


@pytest.fixture
def lib(monkeypatch):
    r = Recorder(codec.lib())
    for m in (codec, batch):
        monkeypatch.setattr(m, "lib", lambda: r)
        monkeypatch.setattr(m, "_stream_handle", lambda: ctypes.c_void_p(0))
    monkeypatch.setattr(batch, "BatchPlan", lambda h, keep, outs=None, staged=False, **kw: SimpleNamespace(keep=keep, outs=outs))
    return r


def stream(short):
    off = codec._index_size_offset(N, L, T)
    ix = torch.zeros(off + 32 if short else codec.index_bytes(N, L, T), dtype=torch.uint8)
    data = torch.zeros(codec.worst_case_bytes(N, L, T), dtype=torch.uint8)
    return codec.DeviceStream(device(data), device(ix), N, L, T)


def test_index_grew():
    assert codec.index_bytes(N, L, T) > codec._index_size_offset(N, L, T) + 32


def roomy(s):
    return s.index.numel() >= codec.index_bytes(N, L, T)


def test_compress_into_a_short_index(lib):
    out = stream(True)
    s = codec.compress(device(torch.zeros(N)), EB, L, T, out=out, ws=WS)
    assert s is out and roomy(out)
    (name, a), = lib.calls
    assert name == "zccl_compress_dev" and a[7].value == out.index.data_ptr()


def test_sum_into_a_short_index(lib):
    out = stream(True)
    s = codec.homsum([stream(False), stream(False)], out=out, ws=WS, stage=False)
    assert s is out and roomy(out)
    (name, a), = lib.calls
    assert name == "zccl_homsum_dev" and a[8].value == out.index.data_ptr()


def test_plans_into_a_short_index(lib):
    xs, outs = [device(torch.zeros(N)) for _ in range(2)], [stream(True), stream(False)]
    batch.compress_plan(xs, [EB, EB], outs)
    sums = [stream(True), stream(False)]
    batch.homsum_plan([[stream(False)] * 2] * 2, sums)
    for (name, a), o, at in zip(lib.calls, (outs, sums), (8, 9)):
        assert all(roomy(s) for s in o), name
        assert list(a[at]) == [s.index.data_ptr() for s in o], name


def test_a_full_index_stays(lib):
    out = stream(False)
    ix = out.index
    codec.compress(device(torch.zeros(N)), EB, L, T, out=out, ws=WS)
    assert out.index is ix


def test_a_short_input_is_indexed_on_the_callers_workspace(lib):
    """What its parse finds wrong is reported where the call's errors are."""
    codec.decompress(stream(True), EB, out=torch.zeros(N), ws=WS)
    codec.homsum([stream(True), stream(False)], out=stream(False), ws=WS, stage=False)
    names = [name for name, _ in lib.calls]
    assert names == ["zccl_parse_dev", "zccl_decompress_dev", "zccl_parse_dev", "zccl_homsum_dev"]
    for (name, a), at in zip(lib.calls, (7, 7, 7, 10)):
        assert a[at].value == WS.ptr.value, name
