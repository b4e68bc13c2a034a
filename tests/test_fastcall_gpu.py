"""The native per-call path of pimaicompiler_amd.ops (cpp/ops_fastcall.cpp) against the Python bodies behind it: the same
results, bit for bit, and the same shapes for every rank, layout and option it takes; None, and with it the Python body's own
checks, for everything else."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class NoNative:
    """Stands in for the extension module: every call falls through to the Python body."""

    def __init__(self, real):
        self.real = real

    def __getattr__(self, name):
        if name.startswith("fast_"):
            return lambda *args: None
        return getattr(self.real, name)


def both(monkeypatch, call):
    """(native path's result, Python body's result) of one call."""
    from pimaicompiler_amd import ops as O
    real = O._native()
    a = call()
    with monkeypatch.context() as m:
        m.setattr(O, "_native_module", NoNative(real))
        b = call()
    return a, b


def same(a, b):
    if isinstance(a, (tuple, list)):
        assert len(a) == len(b)
        for p, q in zip(a, b):
            same(p, q)
    else:
        assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a, b)


def half(*shape):
    return (0.1 * torch.randn(*shape)).half().to(DEV)


@pytest.mark.parametrize("a,b", [
    ((1, 24), (24, 40)), ((1, 1, 24), (24, 40)), ((1, 1, 1, 24), (24, 40)), ((1, 24), (1, 1, 24, 40)), ((40, 24), (24, 1)),
    ((1, 40, 24), (24, 1)), ((40, 24), (1, 24, 1)), ((24,), (24, 40)), ((40, 24), (24,)), ((1, 7), (7, 1)), ((3, 24), (24, 40)), ((24, 24), (24, 1))])
@pytest.mark.parametrize("layout", ["dense", "transposed", "pitched"])
def test_products_of_every_rank_and_layout(ops, monkeypatch, a, b, layout):
    torch.manual_seed(len(a) * 10 + len(b))

    def lay(t):
        if layout == "transposed" and t.dim() >= 2:
            return t.transpose(-1, -2).contiguous().transpose(-1, -2)
        if layout == "pitched" and t.dim() >= 2:
            wide = torch.zeros(*t.shape[:-1], t.size(-1) + 8, dtype=torch.float16, device=DEV)
            wide[..., :t.size(-1)] = t
            return wide[..., :t.size(-1)]
        return t
    x, y = lay(half(*a)), lay(half(*b))
    same(*both(monkeypatch, lambda: ops.custom_aten_matmul(x, y)))
    if len(a) >= 2 and len(b) >= 2 and not (a[-2] == 1 and b[-1] == 1) and (a[-2] == 1 or b[-1] == 1):
        bias = half(b[-1] if a[-2] == 1 else a[-2])
        for act in ("none", "aten::relu"):
            same(*both(monkeypatch, lambda: ops.custom_aten_addmm(act, bias, x, y)))


def test_linear_group_and_projection(ops, monkeypatch):
    w, b = half(40, 24), half(40)
    for x in (half(24), half(1, 24), half(1, 1, 24)):
        same(*both(monkeypatch, lambda: ops.aten_linear(x, w, b, "aten::relu")))
        same(*both(monkeypatch, lambda: ops.aten_linear(x, w)))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    got = ops.aten_linear(x, w, b, stream=side)
    side.synchronize()
    same(got, ops.aten_linear(x, w, b))
    ws = [half(40, 24), half(33, 24), half(8, 64)]
    xs, bs = [half(1, 24), half(24), half(1, 64)], [half(40), None, half(8)]
    same(*both(monkeypatch, lambda: ops.execute_gemv_group(xs, ws, bs, ["none", "aten::relu", "none"])))
    same(*both(monkeypatch, lambda: ops.execute_gemv_group(tuple(xs), tuple(ws))))
    x2, bias = half(17, 24), torch.randn(40, device=DEV)
    same(*both(monkeypatch, lambda: ops.input_projection(x2, w, bias)))
    packed = ops.pack_projection_weight(w)
    same(*both(monkeypatch, lambda: ops.input_projection_packed(x2, packed, 40)))


@pytest.mark.parametrize("layers,bidir,T,batch_first,res", [(1, False, 1, False, None), (2, True, 5, True, None), (2, False, 7, False, 1)])
def test_lstm(ops, monkeypatch, layers, bidir, T, batch_first, res):
    from pimaicompiler_amd import workloads
    I = H = 64
    params, x, h0, c0 = workloads.lstm_inputs(3, I, H, layers, bidir, T)
    params, h0, c0 = [p.to(DEV) for p in params], h0.to(DEV), c0.to(DEV)
    x = x.to(DEV).transpose(0, 1).contiguous() if batch_first else x.to(DEV)

    def call():
        return ops.aten_lstm1(x, (h0, c0), params, True, layers, 0.0, False, bidir, batch_first, first_residual_layer=res)
    call()                                                  # (automatic mode measures on the first call)
    a, b = both(monkeypatch, call)
    same(a, b)
    params[0].mul_(0.5)                                     # an in-place update is seen
    assert not torch.equal(call()[0], a[0])
    if res is not None:                                     # one cached plan, with and without the residual sum
        plain = ops.aten_lstm1(x, (h0, c0), params, True, layers, 0.0, False, bidir, batch_first)
        assert not torch.equal(plain[0], call()[0])


def test_what_the_native_path_does_not_take_is_refused_as_before(ops):
    x, w = half(1, 24), half(40, 24)
    with pytest.raises(ops.NNRuntimeException, match="fp16"):
        ops.aten_linear(x.float(), w)
    with pytest.raises(ops.NNRuntimeException, match="GPU"):
        ops.aten_linear(x.cpu(), w)
    with pytest.raises(ops.NNRuntimeException, match="bias has"):
        ops.aten_linear(x, w, half(39))
    with pytest.raises(ops.NNRuntimeException, match="differ in length"):
        ops.execute_gemv_group([x], [w, w])
    with pytest.raises(ops.NNRuntimeException, match="in_w % 8|multiples of 8|grouped launch"):
        ops.execute_gemv_group([half(1, 20)], [half(8, 20)])


def test_a_bias_shorter_than_its_product_is_refused_in_a_group(ops, monkeypatch):
    xs, ws = [half(1, 24), half(1, 24)], [half(40, 24), half(33, 24)]

    def call(*biases):
        return lambda: ops.execute_gemv_group(xs, ws, list(biases))
    same(*both(monkeypatch, call(half(40), half(34))))     # (a longer one's tail is not read)
    from pimaicompiler_amd import ops as O
    for module in (O._native(), NoNative(O._native())):
        monkeypatch.setattr(O, "_native_module", module)
        with pytest.raises(ops.NNRuntimeException, match="bias has 32 elements, the GEMV produces 33"):
            call(None, half(32))()
        with pytest.raises(ops.NNRuntimeException, match="bias has 1 elements, the GEMV produces 40"):
            call(half(1), half(33))()


def test_an_argument_of_the_wrong_kind_reaches_the_python_body(ops, monkeypatch):
    """... whose exception is the caller's, not a SystemError about one left behind by the native call."""
    import ctypes
    x, w = half(5, 24), half(40, 24)
    packed = ops.pack_projection_weight(w)
    for n_out in (40.0, 1 << 70):
        with pytest.raises((ctypes.ArgumentError, TypeError, OverflowError, ops.NNRuntimeException)):
            ops.input_projection_packed(x, packed, n_out)
    with pytest.raises((ctypes.ArgumentError, TypeError, ValueError)):
        ops.aten_linear(x[:1], w, stream="main")


def test_activations_of_a_group_from_a_generator(ops, monkeypatch):
    xs, ws, acts = [half(1, 24), half(1, 24)], [half(40, 24), half(33, 24)], ["none", "aten::relu"]
    native, body = both(monkeypatch, lambda: ops.execute_gemv_group(xs, ws, None, (a for a in acts)))
    same(native, body)
    assert bool((body[1] >= 0).all()) and bool((body[0] < 0).any())
