"""The per-XCD recurrence (mode 4) with both of its kinds of products, v_dot2 and sparse matrix instructions: whole fragments and ragged
ones.  Every test asks which kind its size takes (lstm_kinds.py), so that a move of the lines cannot leave one of them untested."""
import pytest
import torch

from lstm_kinds import on_dot

from oracle import oracle
from pimaicompiler_amd import workloads

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# (hidden size, steps)
ONE_SPARSE = [(384, 40), (392, 40), (392, 31), (512, 32), (520, 33), (640, 100), (648, 95), (648, 96), (768, 96), (776, 47), (776, 48), (896, 48), (904, 15),
              (904, 16), (1024, 16), (256, 20)]
ONE_DOT = [(8, 12), (56, 40), (64, 7), (128, 7), (392, 6), (512, 4), (520, 10), (640, 10), (776, 6), (904, 5), (1024, 6)]
STACK_SPARSE = [(128, 12), (136, 9), (136, 10), (512, 10), (520, 23), (520, 24), (640, 24), (648, 9), (648, 10), (1024, 10)]


def plan_of(ops, params, layers, bidir, T, res=None):
    plan = ops.LstmPlan([p.to(DEV) for p in params], True, layers, bidir, T)
    plan.set_mode(4)
    if res is not None:
        plan.set_residual(res)
    return plan


@pytest.mark.parametrize("bidir", [False, True])
@pytest.mark.parametrize("H,T", ONE_SPARSE + ONE_DOT)
def test_every_step_is_as_close_to_64_bits_as_its_sums_allow(ops, H, T, bidir):
    """h of every step against float64 arithmetic on the previous h the kernel itself made, with the cell state carried in float64.
    A pre-activation of K = I + H products is off by at most (K / 8 + 8) * 2^-24 of the sum of their magnitudes (eight and more
    are summed before a rounding), the activations by a few ulps of fp32 (2^-21), c by what its steps add up, and h is
    rounded to fp16 once."""
    I, D = 40, 2 if bidir else 1
    params, x, h0, c0 = workloads.lstm_inputs(H + T, I, H, 1, bidir, T)
    g = torch.Generator().manual_seed(H)
    h0, c0 = (0.3 * torch.randn(h0.shape, generator=g)).half(), (0.3 * torch.randn(c0.shape, generator=g)).half()
    plan = plan_of(ops, params, 1, bidir, T)
    xd = x.reshape(T, I).to(DEV)
    y, hn, cn = plan.forward(xd, h0.to(DEV), c0.to(DEV))
    plan.status()
    assert all(torch.equal(a, b) for a, b in zip((y, hn, cn), plan.forward(xd, h0.to(DEV), c0.to(DEV))))   # the same bits again
    for d in range(D):
        w_ih, w_hh, b_ih, b_hh = (p.to(DEV).double() for p in params[4 * d:4 * d + 4])
        yd = y.view(T, D, H)[:, d].double()
        xs = xd.double()
        if d:
            yd, xs = yd.flip(0), xs.flip(0)
        prev = torch.cat([h0.to(DEV).double().view(D, H)[d:d + 1], yd[:-1]])
        a = xs @ w_ih.t() + prev @ w_hh.t() + b_ih + b_hh
        size = xs.abs() @ w_ih.abs().t() + prev.abs() @ w_hh.abs().t() + (b_ih + b_hh).abs()
        off = (((I + H) / 8 + 8) * 2.0 ** -24 * size).view(T, 4, H).amax(1) + 2.0 ** -21
        i, f, u, o = a.chunk(4, 1)
        c, bound = c0.to(DEV).double().view(D, H)[d], torch.zeros(H, dtype=torch.float64, device=DEV)
        for t in range(T):
            c = torch.sigmoid(f[t]) * c + torch.sigmoid(i[t]) * torch.tanh(u[t])
            bound = bound + 3 * off[t]              # f' |c|, i' |g| and i g' are each at most one off
            want = torch.sigmoid(o[t]) * torch.tanh(c)
            assert bool(((yd[t] - want).abs() <= want.abs() * 2.0 ** -11 + 2.0 ** -25 + bound + off[t]).all()), t
        assert bool(((cn.view(D, H)[d].double() - c).abs() <= c.abs() * 2.0 ** -11 + 2.0 ** -25 + bound).all())
        assert torch.equal(hn.view(D, H)[d].double(), yd[-1])


@pytest.mark.parametrize("layers,res", [(2, None), (3, 1), (4, None)])
@pytest.mark.parametrize("H,T", STACK_SPARSE)
def test_stacks_match_libtorch(ops, H, T, layers, res):
    params, x, h0, c0 = workloads.lstm_inputs(H + T, H if res is not None else 40, H, layers, False, T)
    plan = plan_of(ops, params, layers, False, T, res)
    xd = x.reshape(T, -1).to(DEV)
    y, hn, cn = plan.forward(xd, h0.to(DEV), c0.to(DEV))
    plan.status()
    if res is None:
        want = oracle.torch_lstm(x, h0, c0, params, True, layers, False)
    else:
        step = ops.LstmPlan([p.to(DEV) for p in params], True, layers, False, T)
        step.set_mode(1)
        step.set_residual(res)
        want = step.forward(xd, h0.to(DEV), c0.to(DEV))
    for got, w in zip((y, hn, cn), want):
        assert float((got.float().cpu().reshape(-1) - w.float().cpu().reshape(-1)).abs().max()) <= 5e-3


@pytest.mark.parametrize("H,T,layers,bidir,res,dot", [
    (128, 12, 2, False, None, False), (128, 12, 3, False, 1, False), (256, 12, 1, True, None, False), (392, 32, 1, False, None, False),
    (904, 16, 1, True, None, False), (136, 12, 2, False, None, False), (520, 24, 3, False, 1, False),
    (392, 6, 1, True, None, True), (520, 10, 1, True, None, True), (640, 10, 1, False, None, True), (1024, 6, 1, False, None, True),
    (56, 12, 2, False, None, True), (16, 12, 3, False, None, True), (640, 6, 2, False, None, True), (1024, 3, 2, False, None, True)])
def test_waits_that_give_up_and_nans_in_both_kinds(ops, H, T, layers, bidir, res, dot):
    assert dot == (res is None and on_dot(H, T, 1 if bidir else layers))
    params, x, h0, c0 = workloads.lstm_inputs(H, H, H, layers, bidir, T)
    plan = plan_of(ops, params, layers, bidir, T, res)
    args = (x.reshape(T, H).to(DEV), h0.to(DEV), c0.to(DEV))
    want = plan.forward(*args)
    plan.set_spin_limit(0)
    for _ in range(20):                                    # (two directions of 256: in a forward of 20 every first look finds its word)
        got = plan.forward(*args)
        plan.status()
        for a, b in zip(got, want):                        # right whether or not a wait gave up in it
            assert float((a.float() - b.float()).abs().max()) <= 2e-3
        if plan.fallbacks()[0]:
            break                                          # every workgroup made its units by itself
    assert plan.fallbacks()[0] == 1
    plan.set_spin_limit(1 << 22)
    again = plan.forward(*args)
    assert all(torch.equal(a, b) for a, b in zip(again, want))
    bad = args[0].clone()
    at = T // 2
    bad[at, 3] = float("nan")
    y = plan.forward(bad, args[1], args[2])[0]
    plan.status()
    assert plan.fallbacks()[0] == 1                        # nobody waits for a value that is a NaN
    if bidir:
        fwd, bwd = y[:, :H], y[:, H:]
        assert bool(torch.isnan(fwd[at:]).all()) and bool(torch.isnan(bwd[:at + 1]).all())
        assert torch.equal(fwd[:at], want[0][:at, :H]) and torch.equal(bwd[at + 1:], want[0][at + 1:, H:])
    else:
        assert bool(torch.isnan(y[at:]).all()) and torch.equal(y[:at], want[0][:at])


@pytest.mark.parametrize("H,layers,bidir,short,long", [(512, 1, True, 6, 7), (1024, 1, False, 6, 7), (64, 1, False, 23, 24), (264, 2, False, 3, 4), (640, 2, False, 6, 7)])
def test_one_plan_runs_both_kinds_in_turn(ops, H, layers, bidir, short, long):
    """The two kinds share the exchange, its counters and its slots: sequences on either side of a line in turn, eager and replayed."""
    chained = 1 if bidir else layers
    assert on_dot(H, short, chained) and not on_dot(H, long, chained)
    params, x, h0, c0 = workloads.lstm_inputs(H, 40, H, layers, bidir, long)
    xd, h0, c0 = x.reshape(long, 40).to(DEV), h0.to(DEV), c0.to(DEV)
    want = {T: plan_of(ops, params, layers, bidir, T).forward(xd[:T], h0, c0) for T in (short, long)}
    plan = plan_of(ops, params, layers, bidir, long)
    for T in (short, long, long, short, short, long):
        assert all(torch.equal(a, b) for a, b in zip(plan.forward(xd[:T], h0, c0), want[T]))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        one = plan.forward(xd[:long], h0, c0)
        two = plan.forward(xd[:short], h0, c0)
    for _ in range(3):
        for t in (*one, *two):
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip((*one, *two), (*want[long], *want[short])))
        assert all(torch.equal(a, b) for a, b in zip(plan.forward(xd[:short], h0, c0), want[short]))
    plan.status()
    assert plan.fallbacks() == (0, True)
