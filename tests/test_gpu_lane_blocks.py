"""The lane kernels' block paths at their edges: the FP32 quantizer where it
hands over to the FP64 one (2^23 bounds from zero, NaN, infinities, fractions
around zero), short last blocks of every length, every class of width (below 8,
16, 24, 32, and 32) alone and mixed in a tile, and tiles too wide for half or
the whole of a wave's buffer.  Against the oracle, byte for byte."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu

L = 36


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


def round_trip(codec, x, eb, T):
    d = torch.from_numpy(x).cuda()
    s = codec.compress(d, eb, L, T)
    y = codec.decompress(s, eb)
    torch.cuda.synchronize()
    codec.check_errors()
    cx = O.compress(x, eb, L, T)
    assert np.array_equal(s.to_host(), cx)
    assert np.array_equal(y.cpu().numpy().view(np.uint32), O.decompress(cx, x.size, eb, L, T).view(np.uint32))
    return s, cx


@pytest.mark.parametrize("eb", [1.0, 0.3, 1e-30, 1e30])
def test_quantizer_edges(codec, eb):
    say("quantizer", eb)
    rng = np.random.default_rng(8)
    e = np.float32(eb)
    near = np.array([2.0 ** 23 - 1, 2.0 ** 23 - 0.5, 2.0 ** 23, 2.0 ** 23 + 1, 2.0 ** 24 - 1, 2.0 ** 24, 2.0 ** 24 + 2])
    with np.errstate(over="ignore", under="ignore"):
        edge = (np.concatenate([near, -near, [0.0, -0.0, 0.4, -0.4, 0.9999999, -0.9999999, 1.0, -1.0, 1.5, -1.5]])
                .astype(np.float32) * e).astype(np.float32)
        # one tile within the FP32 quantizer, one with the edges, one with what is no number
        a = (rng.integers(-5000, 5000, 2305) / np.float32(7)).astype(np.float32) * e
        b = rng.choice(edge, 2304).astype(np.float32)
        c = a[:2304].copy()
        c[[5, 700, 1800]] = [np.nan, np.inf, -np.inf]
        d = (rng.uniform(-0.99, 0.99, 2304)).astype(np.float32) * e
        tiny = np.full(2304, np.float32(1e-45))
        tiny[::3] *= -1
    round_trip(codec, np.concatenate([a, b, c, d, tiny, a]).astype(np.float32), eb, 1)


@pytest.mark.parametrize("tail", range(1, 37))
def test_short_last_blocks(codec, tail):
    """Segments of 1 + 36 k + tail values at widths below 8, 16 and 24."""
    say("short", tail)
    rng = np.random.default_rng(tail)
    for amp in (20, 3000, 500_000):
        n = 4 * (1 + 36 * 66 + tail)
        x = rng.integers(-amp, amp + 1, n).astype(np.float32)
        s, cx = round_trip(codec, x, 1.0, 4)
        total = codec.homsum([s, s, s], stage=False)
        torch.cuda.synchronize()
        codec.check_errors()
        assert np.array_equal(total.to_host(), O.homsum([cx, cx, cx], n, L, 4))


WIDTHS = {"narrow": [3], "byte": [12], "two": [18], "three": [27], "widest": [31], "low": [1, 7, 8, 15, 16], "all": list(range(32)),
          "half": [16, 17], "full": [30], "rest": [2, 30]}


@pytest.mark.parametrize("name", WIDTHS)
def test_width_classes(codec, knobs, name):
    """Blocks of these widths in turn, in sums of operands alike and unlike,
    in every form of the sum."""
    say("widths", name)
    T, nb = 2, 64 * 5 + 3
    n = T * (1 + 36 * nb - 7)
    rng = np.random.default_rng(len(name))

    def field(ws, shift):
        w = np.repeat([ws[(i + shift) % len(ws)] for i in range(nb * T + 1)], 36)[: n]
        x = np.ldexp(rng.uniform(0.55, 0.95, n), w - 1) * np.where(np.arange(n) % 2, 1.0, -1.0)
        return np.floor(x).astype(np.float32)

    fields = [field(WIDTHS[name], 0), field(WIDTHS[name], 3), field([5], 0), field([0], 0)]
    pairs = [round_trip(codec, x, 1.0, T) for x in fields]
    streams, hosts = [p[0] for p in pairs], [p[1] for p in pairs]
    want = O.homsum(hosts, n, L, T)
    for cfg in ({"layout": 0, "two_pass": 1 << 40}, {"layout": 0, "two_pass": 1}, {"layout": 2}):
        knobs.set_knobs("homsum", cfg)
        total = codec.homsum(streams)
        torch.cuda.synchronize()
        codec.check_errors()
        assert np.array_equal(total.to_host(), want), cfg
