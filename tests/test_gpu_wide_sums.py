"""Sums whose tiles have blocks of width 16 and more: a few of them in a tile of
half a wave's buffer, tiles larger than that, first, last and between narrow
operands, 1 to 32 of them, in every form of the sum.  Against the oracle, byte
for byte; an operand that ends before its tiles is reported in either place."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu

L, T, NB = 36, 2, 64 * 3 + 5
N = T * (1 + L * NB - 9)
FORMS = ({"layout": 0, "two_pass": 1 << 40}, {"layout": 0, "two_pass": 1}, {"layout": 2})


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


@pytest.fixture(scope="module")
def streams(codec):
    """n: narrow; s: some blocks from width 16; w: all of them (and 24, 30)."""
    rng = np.random.default_rng(16)
    out = {}
    for name, widths in {"n": [4], "s": [5] * 9 + [17, 3, 25], "w": [17, 24, 16, 30]}.items():
        w = np.repeat([widths[i % len(widths)] for i in range(NB * T + 1)], L)[:N]
        x = np.floor(np.ldexp(rng.uniform(0.55, 0.95, N), w - 1) * np.where(np.arange(N) % 2, 1.0, -1.0)).astype(np.float32)
        out[name] = (codec.compress(torch.from_numpy(x).cuda(), 1.0, L, T), O.compress(x, 1.0, L, T))
    return out


@pytest.mark.parametrize("order", ["n", "s", "w", "nw", "wn", "ws", "sw", "nsw", "wns", "swwn", "wwss", "nnwnn", "w" * 32,
                                   "wsn" * 10 + "ww", "n" * 31 + "w"])
def test_orders(codec, knobs, streams, order):
    print("[gpu] wide sums", order, flush=True)
    want = O.homsum([streams[c][1] for c in order], N, L, T)
    for cfg in FORMS:
        knobs.set_knobs("homsum", cfg)
        total = codec.homsum([streams[c][0] for c in order])
        torch.cuda.synchronize()
        codec.check_errors()
        assert np.array_equal(total.to_host(), want), cfg


@pytest.mark.parametrize("order", ["wc", "cw", "nc"])
def test_an_operand_that_ends_early(codec, knobs, streams, order):
    """c: w under an index that states half its size."""
    print("[gpu] short operand", order, flush=True)
    w = streams["w"][0]
    ix = w.index.clone()
    ix[w.size_offset: w.size_offset + 8] = torch.tensor([w.size // 2], dtype=torch.int64).view(torch.uint8).cuda()
    cut = codec.DeviceStream(w.data, ix, N, L, T)
    for cfg in FORMS:
        knobs.set_knobs("homsum", cfg)
        ws = codec.Workspace(codec.num_tiles(N, L, T))
        codec.homsum([cut if c == "c" else streams[c][0] for c in order], ws=ws)
        assert ws.errors() == 16, cfg
