"""GEMV operands of any size and address: rows that are no whole 16-byte pieces.  Reference: the float64 product.  Tolerance per output: half an ulp of fp16
(2^-11 of the value, 2^-25 below the normal range) for the one rounding, and (in + 1) * 2^-24 times the sum of the products'
magnitudes for any order of fp32 sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def at_offset(t, off):
    """The same values at an address `off` halves behind a 16-byte boundary."""
    buf = torch.zeros(t.numel() + off + 8, dtype=torch.float16, device=DEV)
    v = buf[off:off + t.numel()].view(t.shape)
    v.copy_(t)
    return v


def call(order, W, x, b, in_w, out_w, ld, relu, off_y=0):
    from pimaicompiler_amd import _lib as L
    lib = L.load()
    y = torch.full((out_w + off_y + 1,), float("nan"), dtype=torch.float16, device=DEV)
    rc = lib.pimhip_execute_gemv(y[off_y:].data_ptr(), x.data_ptr(), W.data_ptr(), b.data_ptr() if b is not None else None, in_w, out_w, ld,
                                 L.PIMHIP_ACT_RELU if relu else L.PIMHIP_ACT_NONE, order, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.pimhip_last_error()
    assert bool(torch.isnan(y[off_y + out_w:]).all()) and bool(torch.isnan(y[:off_y]).all())   # nothing behind or in front of it
    return y[off_y:off_y + out_w]


def check(y, w_out_in, x, b, relu):
    w, xd = w_out_in.double(), x.double()
    want = w @ xd + (b.double() if b is not None else 0)
    size = w.abs() @ xd.abs() + (b.double().abs() if b is not None else 0)
    want = want.relu() if relu else want
    tol = want.abs() * 2.0 ** -11 + 2.0 ** -25 + (w.size(1) + 1) * 2.0 ** -24 * size
    assert bool(((y.double() - want).abs() <= tol).all())


@pytest.mark.parametrize("out_w,in_w,off_w,off_x,pitch", [
    (1, 1, 1, 1, 0), (3, 5, 0, 0, 0), (9, 7, 3, 5, 2), (5, 8, 1, 0, 0), (4, 15, 0, 0, 1), (130, 513, 0, 1, 0), (1023, 2049, 7, 0, 0),
    (1024, 1023, 0, 3, 5), (1025, 1029, 2, 2, 0), (1024, 1024, 1, 0, 0), (1024, 1024, 0, 1, 0), (40, 4103, 0, 0, 0),
    (2049, 4099, 5, 1, 0), (1500, 6151, 0, 0, 0)])   # the last two exceed 16 MB or 4096 columns: other launch shapes and loads
def test_rows_of_any_length_at_any_address(ops, out_w, in_w, off_w, off_x, pitch):
    from pimaicompiler_amd import _lib as L
    g = torch.Generator().manual_seed(out_w + in_w)
    ld = in_w + pitch
    W = at_offset((0.1 * torch.randn(out_w, ld, generator=g)).half(), off_w)
    x = at_offset(torch.randn(in_w, generator=g).half(), off_x)
    b = torch.randn(out_w, generator=g).half().to(DEV)
    for bias, relu in ((b, True), (None, False)):
        check(call(L.PIMHIP_W_X_I, W, x, bias, in_w, out_w, ld, relu, off_w), W[:, :in_w], x, bias, relu)
