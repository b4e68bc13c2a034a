"""Greedy decoding of utterances in chunks of frames on both sides of the line between the kernel for few frames and the one that runs its
first layer for every symbol (rnnt_greedy_every in csrc/rnnt_plan.h), in turn on one plan, eager and replayed from graphs, and with a wait
that gives up.  Against the loop of single steps: same bits."""
import pytest
import torch

from test_rnnt_gpu import DEV, dev
from test_rnnt_greedy_gpu import check, loop_driven_from_the_host, model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,I,H,J,V,chunks", [
    (1, 64, 64, 64, 29, (1, 14, 15, 1, 3)), (1, 320, 72, 64, 64, (31, 32, 1)), (2, 320, 320, 512, 20, (1, 11, 12, 7, 13, 1)), (2, 64, 64, 512, 40, (19, 20, 1)),
    (2, 512, 64, 640, 64, (1, 31, 32, 2)), (2, 320, 64, 64, 128, (63, 64, 1)), (3, 64, 72, 64, 100, (49, 50, 5)), (2, 64, 64, 64, 129, (1, 12, 65)),
])
def test_chunks_on_both_sides_of_the_line(ops, L, I, H, J, V, chunks):
    F, blank, per = 136, V // 3, 3
    params, joint, enc, embedding, x0 = model(11 * V + H + L, L, I, H, F, J, V, sum(chunks), blank, 0.1)
    plan = ops.RnntPlan(dev(params), True, L, tuple(dev(joint)))
    g = torch.Generator().manual_seed(V)
    h, c = (0.3 * torch.randn(L, H, generator=g)).half().to(DEV), torch.randn(L, H, generator=g).half().to(DEV)
    at, first, emitted = 0, True, 0
    for T in chunks:
        frames = enc[at:at + T]
        want = loop_driven_from_the_host(plan, frames, embedding, x0, blank, per, per * T, h, c, first)

        def call():
            return plan.greedy_decode(frames, embedding, x0, blank, per, h0=h, c0=c, run_prediction_first=first)
        emitted += check(call(), want)[0]
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = call()
        for _ in range(3):
            graph.replay()
            check(got, want)
            check(call(), want)
        h, c, at = want[3], want[4], at + T
        if want[5]:           # the chunk's last symbol opens the next one
            x0 = embedding[want[6]]
        first = want[5]
    assert emitted > 0 and plan.fallbacks() == (0, True)
    want = loop_driven_from_the_host(plan, enc[:4], embedding, x0, blank, per, 3 * per, h, c, True)
    plan.set_spin_limit(0)
    for _ in range(20):
        r = check(plan.greedy_decode(enc[:4], embedding, x0, blank, per, max_symbols=3 * per, h0=h, c0=c), want)
        if r[3]:
            break
    assert r[3] == 1 and plan.fallbacks()[0] >= 1


@pytest.mark.parametrize("first", [True, False])
@pytest.mark.parametrize("F", [8, 512, 520, 1024, 1032, 1536, 1544, 2048])
@pytest.mark.parametrize("T", [1, 2, 3, 4, 5, 9])
def test_frames_summed_by_rows_and_by_frames(ops, F, T, first):
    """No more frames than a round asks for and more of them, of every number of 16-byte pieces to a lane, the last of them whole and not."""
    L, H, J, V, blank = 1, 64, 64, 29, 3
    params, joint, enc, embedding, x0 = model(F + T, L, H, H, F, J, V, T, blank, 0.1)
    plan = ops.RnntPlan(dev(params), True, L, tuple(dev(joint)))
    g = torch.Generator().manual_seed(T)
    h, c = (0.3 * torch.randn(L, H, generator=g)).half().to(DEV), torch.randn(L, H, generator=g).half().to(DEV)
    want = loop_driven_from_the_host(plan, enc, embedding, x0, blank, 3, 3 * T, h, c, first)
    for _ in range(2):
        check(plan.greedy_decode(enc, embedding, x0, blank, 3, h0=h, c0=c, run_prediction_first=first), want)
