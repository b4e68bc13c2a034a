"""The decoder step on both sides of the line between weights that stay in the caches from step to step and more than these hold
(csrc/decoder_kernels.h, kDecKeptBytes = 240 MB): only how the rows are read differs, so a step with 121000 classifier rows (265 MB
with the layers' weights) gives the state and, of the first 3000 rows, the logits of one with 3000, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("L", [1, 2])
def test_rows_past_the_caches_give_the_same_bits(ops, L):
    H, V, few = 1024, 121000, 3000
    assert (L * 8 * H * H + few * H) * 2 <= 240 << 20 < (L * 8 * H * H + V * H) * 2
    g = torch.Generator(device=DEV).manual_seed(L)
    rnd = lambda *shape: ((2 * torch.rand(*shape, generator=g, device=DEV) - 1) / 32).half()  # noqa: E731
    params = []
    for l in range(L):
        params += [rnd(4 * H, H if l == 0 else 2 * H), rnd(4 * H, H), rnd(4 * H), rnd(4 * H)]
    w, b = rnd(V, H), rnd(V)
    x, ctx, h, c = rnd(H) * 32, rnd(H) * 32, list(rnd(L, H).unbind(0)), list(rnd(L, H).unbind(0))
    got = []
    for rows in (V, few):
        plan = ops.DecoderPlan(params, True, L, first_takes_context=False, classifier=(w[:rows].contiguous(), b[:rows].contiguous()))
        hn, cn = [torch.empty_like(t) for t in h], [torch.empty_like(t) for t in c]
        logits = torch.empty(rows, dtype=torch.float16, device=DEV)
        plan.bind(x, h, c, ctx=ctx if L > 1 else None, hn=hn, cn=cn, logits=logits)()
        torch.cuda.synchronize()
        got.append((hn, cn, logits))
    assert all(torch.equal(p, q) for p, q in zip(got[0][0] + got[0][1], got[1][0] + got[1][1]))
    assert torch.equal(got[0][2][:few], got[1][2])
    top = got[0][0][-1].float()
    assert float((got[0][2].float() - (w.float() @ top + b.float())).abs().max()) <= 1e-3   # |logits| < 1: half a unit, and fp32 sums
