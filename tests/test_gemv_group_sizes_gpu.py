"""execute_gemv_group at the counts where the size of a launch's arguments changes (4, 8, 16, 32 products) and beyond one launch, with
activations and biases that differ from product to product.  A row of the sums is fp32, the result one rounding to fp16: against the
product in 64 bits at most half a unit in the last place (2^-11 relative) plus the sums' own error, below 1e-4 at 264 columns of
products of at most 1."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("count", [1, 4, 5, 8, 9, 16, 17, 32, 33, 64])
def test_every_product_of_a_group_is_its_own(ops, count):
    g = torch.Generator().manual_seed(count)
    xs = [(torch.rand(1, 264, generator=g) * 2 - 1).half() for _ in range(count)]
    ws = [((torch.rand(7 + 13 * (i % 5), 264, generator=g) * 2 - 1) / 8).half() for i in range(count)]
    bs = [torch.rand(w.size(0), generator=g).half() if i % 3 else None for i, w in enumerate(ws)]
    acts = ["aten::relu" if i % 2 or i == 31 else "none" for i in range(count)]
    got = ops.execute_gemv_group([x.to(DEV) for x in xs], [w.to(DEV) for w in ws], [b.to(DEV) if b is not None else None for b in bs], acts)
    torch.cuda.synchronize()
    assert len(got) == count
    for x, w, b, act, y in zip(xs, ws, bs, acts, got):
        want = w.double() @ x.double().reshape(-1) + (b.double() if b is not None else 0.0)
        if act != "none":
            want = torch.relu(want)
        assert bool(((y.cpu().double() - want).abs() <= want.abs() * 2 ** -11 + 1e-4).all())
