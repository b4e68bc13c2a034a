"""Two steps by a launch each, which makes its projection too for a layer that stands alone: one layer and both directions,
inputs narrower and wider than h, the smallest width, a width of no whole block and one of no sequence kernel; a stack of one
direction, which does not; and the lengths around, which have a measured mode of their own.
"""
import pytest
import torch

from oracle import oracle
from pimaicompiler_amd import workloads

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LSTM_TOL = 5e-3  # the recurrence's tests' own: fp16 h against the oracle's


@pytest.mark.parametrize("I,H,L,bidir", [(8, 8, 1, False), (24, 72, 1, True), (2048, 1024, 1, False), (512, 512, 2, True), (40, 136, 2, False), (520, 2056, 1, True)])
def test_two_steps_by_launches(ops, I, H, L, bidir):
    D = 2 if bidir else 1
    params, x, h0, c0 = workloads.lstm_inputs(I + H, I, H, L, bidir, 2)
    g = torch.Generator().manual_seed(H)
    h0, c0 = (0.3 * torch.randn(L * D, 1, H, generator=g)).half(), torch.randn(L * D, 1, H, generator=g).half()
    want = oracle.torch_lstm(x, h0, c0, params, True, L, bidir)
    plan = ops.LstmPlan([p.to(DEV) for p in params], True, L, bidir, 2)
    plan.set_mode(1)
    for _ in range(2):
        for got, w in zip(plan.forward(x.reshape(2, I).to(DEV), h0.to(DEV), c0.to(DEV)), want):
            assert float((got.cpu().float().reshape(-1) - w.float().reshape(-1)).abs().max()) <= LSTM_TOL


def test_two_steps_are_measured_by_themselves(ops):
    params, x, h0, c0 = workloads.lstm_inputs(3, 64, 64, 1, False, 4)
    plan = ops.LstmPlan([p.to(DEV) for p in params], True, 1, False, 4)
    x, h0, c0 = x.reshape(4, 64).to(DEV), h0.to(DEV), c0.to(DEV)
    plan.forward(x[:2], h0, c0)
    assert plan.measured_mode(2) != 0 and plan.measured_mode(3) == 0 and plan.measured_mode(4) == 0
    plan.forward(x[:3], h0, c0)
    assert plan.measured_mode(3) != 0 and plan.measured_mode(4) == 0


@pytest.mark.parametrize("I,H,L,bidir", [(2056, 2056, 1, True), (64, 2056, 2, True), (6600, 2560, 1, False)])
def test_two_steps_with_a_projection_of_their_own(ops, I, H, L, bidir):
    """W_ih too large to be read by each step: of the only layer, of the second of two, and by the kernel for fewer rows."""
    test_two_steps_by_launches(ops, I, H, L, bidir)
