"""Parsed streams whose segments have as many runs of 64 blocks as one wave of
the carry scan takes in one to four steps, and more (sixteen waves): values
equal the oracle's, which they do only from the right carry before every run."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402
from tests.golden import gen  # noqa: E402

pytestmark = pytest.mark.gpu

L, EB, RUN = 36, 1e-3, 36 * 64


@pytest.mark.parametrize("runs,T,tail", [(1, 300, 0), (63, 1, 0), (64, 3, 2), (65, 1, 0), (128, 2, 1), (255, 1, 0), (256, 1, 0),
                                         (256, 3, 2), (257, 1, 0), (257, 3, 1), (1025, 1, 0)])
def test_values_of_a_parsed_stream(runs, T, tail):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from zccl_amd import codec

    n = T * (1 + RUN * runs - 7) + tail
    print("[gpu] carry scan", runs, T, tail, flush=True)
    cx = O.compress(gen.make("grf", n, 5), EB, L, T)
    y = codec.decompress(codec.upload(cx, n, L, T), EB)
    torch.cuda.synchronize()
    codec.check_errors()
    assert np.array_equal(y.cpu().numpy().view(np.uint32), O.decompress(cx, n, EB, L, T).view(np.uint32))
