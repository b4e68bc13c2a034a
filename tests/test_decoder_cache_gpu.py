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


@pytest.mark.parametrize("L,vocabs", [(1, (8000, 13000, 20000, 40000)), (2, (1000, 13000)), (3, (0, 1000)), (4, (1000, 9000, 40000))])
def test_every_way_to_read_the_rows_gives_the_same_bits(ops, L, vocabs):
    """1024 units with all rows plain, the layers' or the classifier's past the L2s, and all plain again (dec_plain_loads): the same state, and
    the same logits of the rows they share."""
    H = 1024
    g = torch.Generator(device=DEV).manual_seed(7 + L)
    rnd = lambda *shape: ((2 * torch.rand(*shape, generator=g, device=DEV) - 1) / 32).half()  # noqa: E731
    params = []
    for l in range(L):
        params += [rnd(4 * H, H if l == 0 else 2 * H), rnd(4 * H, H), rnd(4 * H), rnd(4 * H)]
    w, b, enc = rnd(max(vocabs), H), rnd(max(vocabs)), rnd(9, H)
    x, h, c = rnd(H) * 32, list(rnd(L, H).unbind(0)), list(rnd(L, H).unbind(0))
    att = torch.softmax(torch.randn(9, generator=g, device=DEV), -1).half()
    got = []
    for rows in vocabs:
        plan = ops.DecoderPlan(params, True, L, first_takes_context=False, classifier=(w[:rows].contiguous(), b[:rows].contiguous()) if rows else None)
        plan.set_encoder(enc)
        hn, cn = [torch.empty_like(t) for t in h], [torch.empty_like(t) for t in c]
        logits = torch.empty(rows, dtype=torch.float16, device=DEV)
        step = plan.bind(x, h, c, att=att, hn=hn, cn=cn, logits=logits if rows else None)
        for _ in range(3):
            step()
        torch.cuda.synchronize()
        got.append((hn + cn, logits))
    for state, logits in got[1:]:
        assert all(torch.equal(p, q) for p, q in zip(state, got[0][0]))
        shared = min(len(logits), len(got[0][1]))
        assert torch.equal(logits[:shared], got[0][1][:shared])
    top = got[-1][0][L - 1].float()
    if L < 3:   # (no sums around the top layer: the classifier takes h)
        assert float((got[-1][1].float() - (w[:len(got[-1][1])].float() @ top + b[:len(got[-1][1])].float())).abs().max()) <= 1e-3
