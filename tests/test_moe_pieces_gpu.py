"""The mixture-of-experts step where the kernel for a size changes (16-byte pieces of a row per lane: 512 / 1024 columns of the first
matrix, 1024 / 2048 / 3072 of the second), with as many rows of the second matrix as wavefronts and with one, and with one and two
words for a polling thread.  Against LibTorch CPU with the tolerance of test_moe_gpu.py: its inputs have the same scale."""
import pytest
import torch

from test_moe_gpu import DEV, TOL, dev, libtorch_cpu, make, maxabs

pytestmark = pytest.mark.gpu


# (1536, 1544 and 1792 / 4096: six and seven rows of the second matrix to a block, more than leave wavefronts enough to poll without one)
@pytest.mark.parametrize("d_model,d_ff", [(512, 1024), (520, 1032), (1024, 2048), (1032, 2056), (512, 3072), (520, 3080), (2048, 8), (8, 4096),
                                          (2048, 4096), (1536, 4096), (1544, 4096), (1792, 4096)])
def test_sizes_on_both_sides_of_a_change_of_kernel(ops, d_model, d_ff):
    g, Wr, br, W1, b1, W2, b2 = make(d_model + d_ff, 3, d_model, d_ff, True, scale=0.5 / max(d_model, 64) ** 0.5)
    plan = ops.MoePlan((Wr.to(DEV), br.to(DEV)), dev(W1), dev(W2), dev(b1), dev(b2))
    x = torch.randn(6, d_model, generator=g).half()
    xd, yd = x.to(DEV), torch.empty(6, d_model, dtype=torch.float16, device=DEV)
    expert = torch.full((6, 1), -1, dtype=torch.int32, device=DEV)
    for i in range(6):                         # one behind the other: both sets of the exchange's slots, several times
        plan.bind(xd[i], yd[i], None, expert[i])()
    torch.cuda.synchronize()
    checked = 0
    for i in range(6):
        _, e, _, y, gap = libtorch_cpu(x[i:i + 1], Wr, br, W1, b1, W2, b2, "aten::relu", False)
        if gap > 2 * TOL:
            assert int(expert[i]) == e and maxabs(yd[i], y) <= TOL
            checked += 1
    assert checked >= 3 and plan.fallbacks() == (0, True)
