"""The greedy decoding loop where its first layer runs for every symbol ahead of the decision: vocabularies on both sides of the rule
(64 symbols with one layer, 128 with more) and of a lane's symbols, odd and single ones, embedding rows of one and two pieces a lane in LDS
and in memory, a first step with and without the prediction network.  Against the loop of single steps: same bits."""
import pytest
import torch

from test_rnnt_gpu import DEV, dev
from test_rnnt_greedy_gpu import check, loop_driven_from_the_host, model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("run_prediction_first", [True, False])
@pytest.mark.parametrize("L,I,H,V", [
    (1, 64, 32, 1), (1, 64, 64, 2), (1, 320, 72, 64), (1, 320, 72, 65),
    (2, 64, 64, 63), (2, 520, 64, 29), (2, 1024, 72, 64), (2, 64, 136, 65), (2, 320, 320, 127), (2, 320, 64, 128), (2, 64, 64, 129),
    (3, 64, 64, 29), (4, 72, 64, 100),
])
def test_the_first_layer_ahead_of_the_decision(ops, L, I, H, V, run_prediction_first):
    F, J, T, blank = 128, 64, 64, V // 2   # (frames enough for every one of these vocabularies)
    params, joint, enc, embedding, x0 = model(31 * V + H + L, L, I, H, F, J, V, T, blank, 0.1 if V > 2 else -0.3)
    plan = ops.RnntPlan(dev(params), True, L, tuple(dev(joint)))
    g = torch.Generator().manual_seed(V)
    h0 = (0.3 * torch.randn(L, H, generator=g)).half().to(DEV)
    c0 = torch.randn(L, H, generator=g).half().to(DEV)
    want = loop_driven_from_the_host(plan, enc, embedding, x0, blank, 3, 3 * T, h0, c0, run_prediction_first)
    r = check(plan.greedy_decode(enc, embedding, x0, blank, 3, h0=h0, c0=c0, run_prediction_first=run_prediction_first), want)
    assert r[3] == 0 and (V == 1 or r[0] > 0)


@pytest.mark.parametrize("L,J,V", [(2, 512, 32), (2, 520, 32), (2, 1024, 31), (2, 1032, 29), (2, 512, 33), (2, 8, 40), (2, 512, 64), (3, 504, 41),
                                   (2, 520, 64), (1, 512, 29)])
def test_the_decision_behind_a_symbol(ops, L, J, V):
    """Where every block makes it (four or eight rows of W2 a wavefront, one or two pieces of them a lane) and on the other side of that rule."""
    I, H, F, T, blank = 64, 64, 128, 40, 0
    params, joint, enc, embedding, x0 = model(7 * V + J, L, I, H, F, J, V, T, blank, 0.0)
    plan = ops.RnntPlan(dev(params), True, L, tuple(dev(joint)))
    want = loop_driven_from_the_host(plan, enc, embedding, x0, blank, 3, 3 * T)
    r = check(plan.greedy_decode(enc, embedding, x0, blank, 3), want)
    assert r[3] == 0 and r[0] > 0


@pytest.mark.parametrize("L,F,J,V,T,blank_bias", [
    (2, 128, 64, 29, 120, -30.0),    # symbols alone, more of them than the rings hold: nobody waits for the symbol blocks
    (2, 1024, 64, 29, 140, 0.0),     # frames of two pieces a lane, a mix
    (2, 1032, 64, 40, 70, 0.0),      # of three
    (1, 2048, 72, 29, 70, 9.0),      # of four, blanks alone: frames across the ring of their sums
    (2, 8, 64, 64, 130, 9.0),
    (2, 200, 64, 129, 70, 0.0),
])
def test_rings_and_frames(ops, L, F, J, V, T, blank_bias):
    """Frames of every number of pieces, summed ahead in a ring, and hidden vectors' entries used again after runs of one kind of decision."""
    I, H, blank = 64, 64, V - 1
    params, joint, enc, embedding, x0 = model(3 * V + F, L, I, H, F, J, V, T, blank, blank_bias)
    plan = ops.RnntPlan(dev(params), True, L, tuple(dev(joint)))
    want = loop_driven_from_the_host(plan, enc, embedding, x0, blank, 2, 2 * T)
    r = check(plan.greedy_decode(enc, embedding, x0, blank, 2), want)
    assert r[3] == 0 and (r[0] == 2 * T if blank_bias < 0 else r[0] == 0 if blank_bias > 5 else r[0] > 0)
