"""One step of a stack with sums around its layers: the sum is made by the step's launch, with the bits of one layer after the
other and an addition behind each (h is not touched by it).  Widths of one unit's block, of odd blocks, of a lane's edge.
"""
import pytest
import torch

from pimaicompiler_amd import workloads

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("H,L,first", [(8, 1, 0), (72, 5, 0), (136, 3, 1), (1024, 4, 1), (1040, 2, 1), (2056, 3, 2)])
def test_bits_of_a_launch_per_sum(ops, H, L, first):
    params, x, h0, c0 = workloads.lstm_inputs(H, H, H, L, False, 1)
    params = [p.to(DEV) for p in params]
    g = torch.Generator().manual_seed(H)
    x, h0, c0 = x.reshape(1, H).to(DEV), (0.3 * torch.randn(L, H, generator=g)).half().to(DEV), torch.randn(L, H, generator=g).half().to(DEV)
    plan = ops.LstmPlan(params, True, L, False, 1)
    plan.set_residual(first)
    layers = [ops.LstmPlan(params[4 * l:4 * l + 4], True, 1, False, 1) for l in range(L)]
    for _ in range(2):
        y, hn, cn = plan.forward(x, h0, c0)
        cur = x
        for l in range(L):
            out, hl, cl = layers[l].forward(cur, h0[l:l + 1], c0[l:l + 1])
            assert torch.equal(hn.reshape(L, H)[l], hl.reshape(H)) and torch.equal(cn.reshape(L, H)[l], cl.reshape(H))
            cur = (out.reshape(1, H) + cur) if l >= first else out.reshape(1, H)
        assert torch.equal(y.reshape(1, H), cur)
