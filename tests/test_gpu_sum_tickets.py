"""Single-pass sums around the number of tiles from which eight waves share a
ticket (1024): whole and partly filled workgroups, one sum, a uniform batch and
a mixed one.  Against the oracle, byte for byte."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402
from tests.golden import gen  # noqa: E402

pytestmark = pytest.mark.gpu

L, EB, TILE = 36, 1e-3, 36 * 64


@pytest.fixture(scope="module")
def zccl():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from zccl_amd import batch, codec

    torch.cuda.set_device(0)
    return codec, batch


def pair(codec, n):
    xs = [gen.make("grf", n, 70 + i) for i in range(2)]
    return [codec.compress(torch.from_numpy(x).cuda(), EB, L, 1) for x in xs], [O.compress(x, EB, L, 1) for x in xs]


@pytest.mark.parametrize("tiles", [1023, 1024, 1025, 1031, 1032, 1033])
def test_one_sum(zccl, tiles):
    codec, _ = zccl
    n = 1 + TILE * tiles - 5
    print("[gpu] sum tickets", tiles, flush=True)
    assert codec.num_tiles(n, L, 1) == tiles
    ops, hosts = pair(codec, n)
    total = codec.homsum(ops, stage=False)
    torch.cuda.synchronize()
    codec.check_errors()
    assert np.array_equal(total.to_host(), O.homsum(hosts, n, L, 1))


@pytest.mark.parametrize("jobs", [[512, 512], [516, 516], [343, 343, 343], [512, 500], [300, 700, 26], [3, 1022], [1, 1032]])
def test_batches(zccl, jobs):
    codec, batch = zccl
    print("[gpu] sum tickets", jobs, flush=True)
    made = {t: pair(codec, 1 + TILE * t - 5) for t in set(jobs)}
    outs = [codec.empty_stream(1 + TILE * t - 5, L, 1) for t in jobs]
    plan = batch.homsum_plan([made[t][0] for t in jobs], outs)
    assert plan.tiles == sum(jobs)
    ws = codec.Workspace(plan.tiles)
    for _ in range(2):
        plan.launch(ws, stage=False)
    codec.check_errors(ws)
    for t, o in zip(jobs, outs):
        assert np.array_equal(o.to_host(), O.homsum(made[t][1], o.n, L, 1))
