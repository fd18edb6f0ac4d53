"""The index carries of 36-value streams (the quantized value before every run
of 64 blocks of a segment), from each kernel that writes an index: compress and
the homomorphic sum in every layout, the parallel and the serial parse.  Sizes
at the edges of runs, tiles and segments: segments of one value, of 64 blocks
to the value and one more, remainders, many runs."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402
from tests.golden import gen  # noqa: E402

pytestmark = pytest.mark.gpu

L, RUN = 36, 36 * 64
CASES = [(16, 16), (37, 1), (RUN + 1, 1), (RUN + 2, 1), (3 * (RUN + 1) + 2, 3), (4 * RUN * 4 + 5, 4), (300_007, 7),
         (2_400_017, 16)]


def say(*a):
    print("[gpu]", *a, flush=True)


@pytest.fixture(scope="module")
def codec():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from zccl_amd import codec as c

    torch.cuda.set_device(0)
    return c


@pytest.fixture
def knobs():
    from zccl_amd import autotune

    yield autotune
    for op in autotune.OPS:
        autotune.reset(op)


def quantized(x, eb):
    return np.trunc(x.astype(np.float64) * np.float64(np.float32(1) / np.float32(eb))).astype(np.int64)


def expected(q, T):
    """q at the first value of every run: 2304 m values into each segment."""
    n = q.size
    tb = n // T
    segs = [(t * tb, tb) for t in range(T)] + ([(T * tb, n - T * tb)] if n % T else [])
    at = [a + RUN * m for a, ln in segs for m in range(max(1, -(-(ln - 1) // RUN)))]
    return q[at].astype(np.int32)


def carries(s):
    off = s.size_offset + 32
    ix = s.index.cpu().numpy()
    return ix[off: off + 4 * ((ix.size - off) // 4)].view(np.int32)


def check(codec, s, q, T, cx, n, eb):
    want = expected(q, T)
    assert np.array_equal(carries(s)[: want.size], want)
    y = codec.decompress(s, eb)
    torch.cuda.synchronize()
    codec.check_errors()
    assert np.array_equal(y.cpu().numpy().view(np.uint32), O.decompress(cx, n, eb, L, T).view(np.uint32))


@pytest.mark.parametrize("n,T", CASES)
def test_compress_and_parse_carries(codec, knobs, n, T):
    say("carries", n, T)
    eb = 1e-3
    x = gen.make("grf", n, 4)
    q, cx, d = quantized(x, eb), O.compress(x, eb, L, T), torch.from_numpy(x).cuda()
    for cfg in ({"layout": 0}, {"layout": 1, "threads": 512}, {"layout": 1, "threads": 256}):
        knobs.set_knobs("compress", cfg)
        check(codec, codec.compress(d, eb, L, T), q, T, cx, n, eb)
    check(codec, codec.upload(cx, n, L, T), q, T, cx, n, eb)
    t = torch.from_numpy(np.ascontiguousarray(cx)).cuda()
    check(codec, codec.from_bytes(t, n, L, T, ws=codec.Workspace(codec.num_tiles(n, L, T))), q, T, cx, n, eb)


@pytest.mark.parametrize("n,T", CASES)
def test_sum_carries(codec, knobs, n, T):
    say("sum carries", n, T)
    eb, k = 1e-3, 3
    xs = [gen.make("grf", n, 40 + r) for r in range(k)]
    hs = [O.compress(x, eb, L, T) for x in xs]
    q, cx = sum(quantized(x, eb) for x in xs), O.homsum(hs, n, L, T)
    streams = [codec.compress(torch.from_numpy(x).cuda(), eb, L, T) for x in xs]
    for cfg in ({"layout": 0}, {"layout": 2}, {"layout": 1, "threads": 256}, {"layout": 1, "threads": 128}):
        knobs.set_knobs("homsum", cfg)
        check(codec, codec.homsum(streams, stage=False), q, T, cx, n, eb)
    knobs.reset("homsum")
    knobs.set_knobs("homsum", {"layout": 0, "two_pass": 1})
    check(codec, codec.homsum(streams), q, T, cx, n, eb)


def test_short_index_is_rebuilt(codec):
    """A stream whose kept index ends before the carries is indexed again."""
    n, T, eb = 100_003, 4, 1e-3
    say("short index", n, T)
    x = gen.make("grf", n, 9)
    s = codec.compress(torch.from_numpy(x).cuda(), eb, L, T)
    old = codec.DeviceStream(s.data, s.index[: s.size_offset + 32].clone(), n, L, T)
    y = codec.decompress(old, eb)
    total = codec.homsum([old, s])
    torch.cuda.synchronize()
    codec.check_errors()
    cx = O.compress(x, eb, L, T)
    assert np.array_equal(y.cpu().numpy().view(np.uint32), O.decompress(cx, n, eb, L, T).view(np.uint32))
    assert np.array_equal(total.to_host(), O.homsum([cx, cx], n, L, T))
