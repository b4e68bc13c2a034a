"""The greedy decoding loop where the symbol blocks' teams and the looks at several steps' logits can go wrong: few and many teams,
a vocabulary on both sides of what a row of 16 lanes takes, three words of a step per lane, utterances shorter than, as long as
and longer than what is published ahead, and runs of blanks across the rings.  Against the loop of single steps: same bits."""
import pytest

from test_rnnt_gpu import dev
from test_rnnt_greedy_gpu import check, loop_driven_from_the_host, model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,I,H,F,J,V,T,blank_bias", [
    (1, 64, 64, 128, 64, 40, 40, 0.3),        # five symbol blocks: the last that a row of 16 lanes takes
    (1, 64, 64, 128, 64, 41, 40, 0.3),        # six
    (1, 64, 64, 128, 64, 512, 30, 0.3),       # 64 symbol blocks, three teams, three words of a step to a lane
    (2, 320, 320, 1024, 512, 360, 25, 0.3),   # two teams of 45 blocks
    (2, 512, 512, 1032, 896, 120, 25, 0.3),   # one team of 15 blocks; frames of more than two pieces to a lane
    (1, 64, 32, 128, 64, 29, 1, 0.3),
    (1, 64, 32, 128, 64, 29, 8, 9.0),         # blanks alone: as many frames as a batch and its neighbours
    (1, 64, 32, 128, 64, 29, 9, 9.0),
    (1, 64, 32, 128, 64, 29, 10, 9.0),
    (1, 64, 32, 128, 64, 29, 300, 9.0),       # around the rings and the tags' eight bits
    (1, 64, 32, 128, 64, 100, 300, 9.0),
])
def test_teams_of_symbol_blocks_decode_as_single_steps_do(ops, L, I, H, F, J, V, T, blank_bias):
    blank = V - 1
    params, joint, enc, embedding, x0 = model(5 * T + V, L, I, H, F, J, V, T, blank, blank_bias)
    plan = ops.RnntPlan(dev(params), True, L, tuple(dev(joint)))
    check(plan.greedy_decode(enc, embedding, x0, blank, max_symbols_per_frame=3),
          loop_driven_from_the_host(plan, enc, embedding, x0, blank, 3, 3 * T))


@pytest.mark.parametrize("V", [168, 169, 336, 337])
def test_words_of_a_step_per_lane(ops, V):
    """Around the lines between the kernels for one, two and three words of a step's logits to a lane (21 and 42 symbol blocks)."""
    L, H, F, J, T = 1, 64, 128, 64, 40
    params, joint, enc, embedding, x0 = model(V, L, H, H, F, J, V, T, V - 1, 0.3)
    plan = ops.RnntPlan(dev(params), True, L, tuple(dev(joint)))
    check(plan.greedy_decode(enc, embedding, x0, V - 1, max_symbols_per_frame=3),
          loop_driven_from_the_host(plan, enc, embedding, x0, V - 1, 3, 3 * T))
