"""The package with libpimhip.so alone: the LibTorch extension with the native per-call path is an accelerator, not a requirement."""
import sys
import warnings

import pytest
import torch


@pytest.fixture
def without(monkeypatch):
    from pimaicompiler_amd import ops as O
    monkeypatch.setitem(sys.modules, "pimaicompiler_amd._aten_ops_pimhip", None)   # (importing it raises ModuleNotFoundError)
    monkeypatch.setattr(O, "_native_module", None)
    return O


def test_a_missing_extension_is_said_once_and_the_bodies_take_over(without):
    x, w = torch.zeros(1, 8, dtype=torch.float16), torch.zeros(4, 8, dtype=torch.float16)
    with pytest.warns(RuntimeWarning, match="has not been built"), pytest.raises(without.NNRuntimeException, match="GPU"):
        without.aten_linear(x, w)                          # (the body's own check: there is no CPU path)
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        for call in (lambda: without.custom_aten_addmm("none", x, x, w.t()), lambda: without.custom_aten_matmul(x, w.t()),
                     lambda: without.execute_gemv_group([x], [w]), lambda: without.input_projection(x, w),
                     lambda: without.input_projection_packed(x, w, 4)):
            with pytest.raises(without.NNRuntimeException, match="GPU"):
                call()


def test_a_broken_extension_is_not_taken_for_a_missing_one(without, monkeypatch):
    def broken(name):
        raise ModuleNotFoundError("No module named 'something_it_needs'", name="something_it_needs")
    monkeypatch.setattr(without.importlib, "import_module", broken)
    with pytest.raises(ModuleNotFoundError, match="something_it_needs"):
        without.aten_linear(torch.zeros(1, 8), torch.zeros(4, 8))


@pytest.mark.gpu
@pytest.mark.filterwarnings("ignore:.*has not been built")
def test_operators_and_bound_steps_give_the_same_bits(ops, monkeypatch):
    from pimaicompiler_amd import ops as O
    DEV = "cuda:0"
    g = torch.Generator().manual_seed(8)

    def half(*shape, scale=0.1):
        return (scale * torch.randn(*shape, generator=g)).half().to(DEV)

    def lstm(i, h):
        return [half(4 * h, i), half(4 * h, h), half(4 * h), half(4 * h)]
    H, V = 64, 29
    w, x, params = half(40, 64), half(1, 64), lstm(64, 64)
    moe_w = (half(4, H), None), [half(128, H) for _ in range(4)], [half(H, 128) for _ in range(4)]
    dec_w, cls = lstm(H, H) + lstm(2 * H, H), (half(100, H), half(100))
    rnnt_w, joint = lstm(H, H), (half(48, 2 * H), half(48), half(V, 48), half(V))
    enc, att, state = half(5, H), torch.softmax(half(5).float(), 0).half(), half(2, H)

    def run():
        out = [O.aten_linear(x, w), O.custom_aten_matmul(x, w.t())]
        out += O.aten_lstm1(half_x, (half_s, half_s), params, True, 1, 0.0, False, False, False)
        moe = O.MoePlan(*moe_w)
        out += moe.forward(x.view(-1))
        dec = O.DecoderPlan(dec_w, True, 2, first_takes_context=False, first_residual_layer=1, classifier=cls)
        h, c, logits = state.clone(), state.clone(), torch.empty(100, dtype=torch.float16, device=DEV)
        dec.set_encoder(enc)
        dec.bind(x.view(-1), list(h.unbind(0)), list(c.unbind(0)), att=att, logits=logits)()
        rnnt = O.RnntPlan(rnnt_w, True, 1, joint)
        hn, cn, sym = torch.empty(1, H, dtype=torch.float16, device=DEV), torch.empty(1, H, dtype=torch.float16, device=DEV), torch.empty(V, dtype=torch.float16, device=DEV)
        rnnt.bind(x.view(-1), state[:1], state[1:], enc[0], hn, cn, sym)(torch.cuda.current_stream())
        torch.cuda.synchronize()
        return out + [h, c, logits, hn, cn, sym]
    half_x, half_s = half(3, 1, 64), half(1, 1, 64)
    run()                                                  # (automatic mode measures on the first call)
    native = run()
    monkeypatch.setitem(sys.modules, "pimaicompiler_amd._aten_ops_pimhip", None)
    monkeypatch.setattr(O, "_native_module", None)
    got = run()
    assert type(O._native()).__name__ == "_WithoutExtension"
    assert len(got) == len(native) and all(torch.equal(a, b) for a, b in zip(got, native))
