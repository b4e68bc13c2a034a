"""The decoder step on both sides of the line between weights that stay in the caches from step to step and more than these hold
(csrc/decoder_plan.h, kDecKeptBytes = 240 MB): only how the rows are read differs, so a step with 121000 classifier rows (265 MB
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


@pytest.mark.parametrize("vocab", [0, 16000])
def test_a_wide_first_layer_past_the_caches(ops, vocab):
    """A first layer over 33000 inputs (274 MB of layers: plain loads, with 16000 classifier rows non-temporal) and over 36864 (310 MB:
    non-temporal), each next to h in 64 bits: a lane adds K / 32 products' sums of two and eight partial sums meet, so a gate's sum
    is off by at most (K / 32 + 16) 2^-24 of the sum of its products' magnitudes, h by that and its rounding to fp16."""
    H = 1024
    for I in (33000, 36864):
        g = torch.Generator(device=DEV).manual_seed(I)
        rnd = lambda *shape: ((2 * torch.rand(*shape, generator=g, device=DEV) - 1) / 64).half()  # noqa: E731
        params = [rnd(4 * H, I), rnd(4 * H, H), rnd(4 * H), rnd(4 * H)]
        x, h, c = rnd(I) * 64, rnd(H) * 64, rnd(H) * 64
        got = []
        for rows in sorted({0, vocab}):
            cls = (rnd(rows, H), rnd(rows)) if rows else None
            plan = ops.DecoderPlan(params, True, 1, first_takes_context=False, classifier=cls)
            hn, cn = torch.empty_like(h), torch.empty_like(c)
            logits = torch.empty(rows, dtype=torch.float16, device=DEV) if rows else None
            plan.bind(x, [h], [c], hn=[hn], cn=[cn], logits=logits)()
            torch.cuda.synchronize()
            got.append((hn, cn))
        assert all(torch.equal(p, q) for p, q in zip(got[0], got[-1]))
        w_ih, w_hh, b_ih, b_hh = (p.double() for p in params)
        a = w_ih @ x.double() + w_hh @ h.double() + b_ih + b_hh
        size = (w_ih.abs() @ x.double().abs() + w_hh.abs() @ h.double().abs()).max()
        off = ((I + H) / 32 + 16) * 2.0 ** -24 * float(size)
        i, f, u, o = a.chunk(4)
        want_c = torch.sigmoid(f) * c.double() + torch.sigmoid(i) * torch.tanh(u)
        want = torch.sigmoid(o) * torch.tanh(want_c)
        hn, cn = got[0]
        bound = 4 * off + 2.0 ** -20   # c collects three gates' errors, h one more; the activations are a few ulps of fp32 off
        assert float((cn.double() - want_c).abs().max()) <= bound + 2.0 ** -11 * float(want_c.abs().max())
        assert float((hn.double() - want).abs().max()) <= bound + 2.0 ** -12
