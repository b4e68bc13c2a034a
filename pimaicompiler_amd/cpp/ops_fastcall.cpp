// The per-call path of pimaicompiler_amd.ops in native code: argument checks, shape dispatch, output tensors and the C ABI call
// of the operators that a decoding loop or an interpreter calls once per token, without a Python object per step.
//
// Each function returns the result, or None where the call is not the plain case (operands that are not fp16 GPU tensors,
// a shape class that goes to LibTorch, a device that has not been initialised): the Python body then takes the call from its
// start, with its own checks and messages.  An error of the C ABI itself is returned as its integer status.
#include "ops_fastcall.h"

#include <torch/extension.h>

#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <vector>

#include "../../include/pimhip.h"

namespace
{
PyObject* none() { Py_RETURN_NONE; }

bool tensorOf(PyObject* o, const at::Tensor*& t)
{
    if (!THPVariable_Check(o)) return false;
    t = &THPVariable_Unpack(o);
    return t->defined() && t->is_cuda() && t->scalar_type() == at::kHalf && t->layout() == at::kStrided && t->dim() <= 4;
}

// The stream a call runs on: an integer handle, or torch's current stream for None.
bool streamOf(PyObject* o, void*& s)
{
    if (o == Py_None) {
        s = static_cast<void*>(c10::hip::getCurrentHIPStream().stream());
        return true;
    }
    if (!PyLong_Check(o)) return false;
    s = PyLong_AsVoidPtr(o);
    if (!PyErr_Occurred()) return true;
    PyErr_Clear();
    return false;
}

// An argument that is no integer of 64 bits is the Python body's to refuse.
bool intOf(PyObject* o, int64_t& v)
{
    v = PyLong_AsLongLong(o);
    if (v != -1 || !PyErr_Occurred()) return true;
    PyErr_Clear();
    return false;
}

at::Tensor newHalf(at::IntArrayRef shape, const at::Tensor& like)
{
    return at::detail::empty_cuda(shape, at::kHalf, like.device(), c10::nullopt);
}

PyObject* status(int rc) { return rc == PIMHIP_ERR_NOT_INITIALIZED ? none() : PyLong_FromLong(rc); }

// The last two dims of `w` as a rows x cols matrix usable where it lies: its own order or (flipped) the other one on the same
// bytes, with the pitch in memory; false: a copy would be needed.
bool weightWhereItLies(const at::Tensor& w, int64_t rows, int64_t cols, bool& flipped, int64_t& ld)
{
    const int64_t d = w.dim();
    const int64_t sr = d >= 2 ? w.stride(d - 2) : cols, sc = w.stride(d - 1);
    flipped = false;
    if ((sc == 1 || cols == 1) && (rows == 1 || sr >= cols)) {
        ld = rows > 1 ? sr : cols;
        return true;
    }
    if ((sr == 1 || rows == 1) && (cols == 1 || sc >= rows)) {
        flipped = true;
        ld = cols > 1 ? sc : rows;
        return true;
    }
    return false;
}

// y = act(weight . x + bias) on `stream`, shaped `shape`; weight is [in, out] for I_X_W and [out, in] for W_X_I.
PyObject* gemv(at::IntArrayRef shape, const at::Tensor& x, const at::Tensor& w, const at::Tensor* bias, int64_t in_w, int64_t out_w,
               int order, int act, void* stream)
{
    bool flipped = false;
    int64_t ld = 0;
    const bool mv = order == PIMHIP_W_X_I;
    if (x.numel() != in_w || w.numel() != in_w * out_w || !x.is_contiguous()) return none();
    if (bias && (bias->numel() != out_w || !bias->is_contiguous())) return none();
    if (!weightWhereItLies(w, mv ? out_w : in_w, mv ? in_w : out_w, flipped, ld)) return none();
    if (flipped) order = mv ? PIMHIP_I_X_W : PIMHIP_W_X_I;
    at::Tensor y = newHalf(shape, w);
    if (y.numel() != out_w) return none();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = pimhip_execute_gemv(y.data_ptr(), x.data_ptr(), w.data_ptr(), bias ? bias->data_ptr() : nullptr, in_w, out_w, ld, act, order, stream);
    Py_END_ALLOW_THREADS
    return rc == PIMHIP_OK ? THPVariable_Wrap(std::move(y)) : status(rc);
}

// PIMHIP_GEMM_* of two operands by the reference's rules (utils.cpp:293-396); PIMHIP_GEMM_UNKNOWN where they do not classify.
int classify(const at::Tensor& a, const at::Tensor& b)
{
    int64_t s1[4] = {0, 0, 0, 0}, s2[4] = {0, 0, 0, 0};
    int r1 = (int)a.dim(), r2 = (int)b.dim(), t = PIMHIP_GEMM_UNKNOWN;
    if (r1 < 1 || r2 < 1) return PIMHIP_GEMM_UNKNOWN;
    for (int i = 0; i < r1; ++i) s1[i] = a.size(i);
    for (int i = 0; i < r2; ++i) s2[i] = b.size(i);
    if (pimhip_gemm_broadcast(s1, &r1, s2, &r2) != PIMHIP_OK || pimhip_get_gemm_type(s1, s2, &t) != PIMHIP_OK) return PIMHIP_GEMM_UNKNOWN;
    return t;
}

// addmm(relu, self, mat1, mat2, stream): customAtenAddmm's VM and MV branches (aten_ops.cpp:626-694)
PyObject* addmm(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    const at::Tensor *self, *a, *b;
    void* stream;
    if (n != 5 || !tensorOf(args[1], self) || !tensorOf(args[2], a) || !tensorOf(args[3], b) || !streamOf(args[4], stream)) return none();
    const int act = args[0] == Py_True ? PIMHIP_ACT_RELU : PIMHIP_ACT_NONE;
    const int64_t d0 = a->dim(), d1 = b->dim();
    const int type = classify(*a, *b);
    if (type == PIMHIP_GEMM_VM && d0 > 1 && d1 > 1) {
        const int64_t out_w = b->size(d1 - 1), in_w = b->size(d1 - 2);
        at::DimVector shape(a->sizes());
        shape[d0 - 1] = out_w;
        shape[d0 - 2] = 1;
        return gemv(shape, *a, *b, self, in_w, out_w, PIMHIP_I_X_W, act, stream);
    }
    if (type == PIMHIP_GEMM_MV && d1 > 1 && d0 > 1) {
        const int64_t out_w = a->size(d0 - 2), in_w = a->size(d0 - 1);
        at::DimVector shape(b->sizes());
        shape[d1 - 1] = 1;
        shape[d1 - 2] = out_w;
        return gemv(shape, *b, *a, self, in_w, out_w, PIMHIP_W_X_I, act, stream);
    }
    return none();
}

// matmul(self, other, stream): customAtenMatmul's VM and MV branches (aten_ops.cpp:770-840)
PyObject* matmul(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    const at::Tensor *a, *b;
    void* stream;
    if (n != 3 || !tensorOf(args[0], a) || !tensorOf(args[1], b) || !streamOf(args[2], stream)) return none();
    const int64_t d0 = a->dim(), d1 = b->dim();
    const int type = classify(*a, *b);
    if (type == PIMHIP_GEMM_VM && d1 > 1 && (d1 > d0 || d0 > 1)) {
        const int64_t out_w = b->size(d1 - 1), in_w = b->size(d1 - 2);
        const int64_t d = d1 > d0 ? d1 : d0;
        at::DimVector shape(d1 > d0 ? b->sizes() : a->sizes());
        shape[d - 1] = out_w;
        shape[d - 2] = 1;
        return gemv(shape, *a, *b, nullptr, in_w, out_w, PIMHIP_I_X_W, PIMHIP_ACT_NONE, stream);
    }
    if (type == PIMHIP_GEMM_MV && d0 > 1 && (d0 > d1 || d1 > 1)) {
        const int64_t out_w = a->size(d0 - 2), in_w = a->size(d0 - 1);
        at::DimVector shape(d0 > d1 ? a->sizes() : b->sizes());
        if (d0 > d1) {
            shape[d0 - 2] = out_w;
            shape.pop_back();
        } else {
            shape[d1 - 1] = 1;
            shape[d1 - 2] = out_w;
        }
        return gemv(shape, *b, *a, nullptr, in_w, out_w, PIMHIP_W_X_I, PIMHIP_ACT_NONE, stream);
    }
    return none();
}

// linear(relu, input, weight, bias or None, stream): one input row on W's own row-major bytes (aten_ops.cpp:304-307)
PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    const at::Tensor *x, *w, *b = nullptr;
    void* stream;
    if (n != 5 || !tensorOf(args[1], x) || !tensorOf(args[2], w) || !streamOf(args[4], stream)) return none();
    if (args[3] != Py_None && !tensorOf(args[3], b)) return none();
    if (w->dim() != 2 || x->dim() < 1 || x->numel() != w->size(1)) return none();
    at::DimVector shape(x->sizes());
    shape.back() = w->size(0);
    return gemv(shape, *x, *w, b, w->size(1), w->size(0), PIMHIP_W_X_I, args[0] == Py_True ? PIMHIP_ACT_RELU : PIMHIP_ACT_NONE, stream);
}

// group(inputs, weights, biases or None, acts (tuple of ints) or None, stream): sibling MV products in one launch
PyObject* group(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    void* stream;
    if (nargs != 5 || !PyList_Check(args[0]) || !PyList_Check(args[1]) || !streamOf(args[4], stream)) return none();
    const Py_ssize_t n = PyList_GET_SIZE(args[1]);
    const bool biases = args[2] != Py_None, acts = args[3] != Py_None;
    if (n < 1 || n > 64 || PyList_GET_SIZE(args[0]) != n || (biases && (!PyList_Check(args[2]) || PyList_GET_SIZE(args[2]) != n)) ||
        (acts && (!PyTuple_Check(args[3]) || PyTuple_GET_SIZE(args[3]) != n)))
        return none();
    void *out[64];
    const void *in[64], *weight[64], *bias[64];
    int64_t in_w[64], out_w[64];
    int act[64];
    std::vector<at::Tensor> y;
    y.reserve((size_t)n);
    for (Py_ssize_t i = 0; i < n; ++i) {
        const at::Tensor *x, *w, *b = nullptr;
        if (!tensorOf(PyList_GET_ITEM(args[0], i), x) || !tensorOf(PyList_GET_ITEM(args[1], i), w)) return none();
        if (biases && PyList_GET_ITEM(args[2], i) != Py_None && !tensorOf(PyList_GET_ITEM(args[2], i), b)) return none();
        if (w->dim() != 2 || x->numel() != w->size(1) || !w->is_contiguous() || !x->is_contiguous() || (b && (!b->is_contiguous() || b->numel() < w->size(0))))
            return none();
        in[i] = x->data_ptr();
        weight[i] = w->data_ptr();
        bias[i] = b ? b->data_ptr() : nullptr;
        in_w[i] = w->size(1);
        out_w[i] = w->size(0);
        act[i] = acts ? (int)PyLong_AsLong(PyTuple_GET_ITEM(args[3], i)) : PIMHIP_ACT_NONE;
        y.push_back(newHalf({out_w[i]}, *w));
        out[i] = y.back().data_ptr();
    }
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = pimhip_execute_gemv_group((int)n, out, in, weight, bias, in_w, out_w, act, stream);
    Py_END_ALLOW_THREADS
    if (rc != PIMHIP_OK) return status(rc);
    PyObject* list = PyList_New(n);
    for (Py_ssize_t i = 0; list && i < n; ++i) PyList_SET_ITEM(list, i, THPVariable_Wrap(std::move(y[(size_t)i])));
    return list;
}

// projection(x, w, bias or None, n_out, packed, stream): out[T, n_out] fp32
PyObject* projection(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    const at::Tensor *x, *w, *b = nullptr;
    void* stream;
    if (n != 6 || !tensorOf(args[0], x) || !tensorOf(args[1], w) || !streamOf(args[5], stream)) return none();
    int64_t n_out;
    if (!intOf(args[3], n_out)) return none();
    if (args[2] != Py_None) {
        if (!THPVariable_Check(args[2])) return none();
        b = &THPVariable_Unpack(args[2]);
        if (!b->is_cuda() || b->scalar_type() != at::kFloat || b->numel() != n_out || !b->is_contiguous()) return none();
    }
    if (x->dim() != 2 || !x->is_contiguous() || !w->is_contiguous()) return none();
    const int64_t T = x->size(0), K = x->size(1);
    const bool packed = args[4] == Py_True;
    if (packed) {
        uint64_t bytes = 0;
        if (pimhip_projection_packed_bytes(K, n_out, &bytes) != PIMHIP_OK || (uint64_t)w->numel() * 2 != bytes) return none();
    } else if (w->dim() != 2 || w->size(0) != n_out || w->size(1) != K) {
        return none();
    }
    at::Tensor out = at::detail::empty_cuda({T, n_out}, at::kFloat, x->device(), c10::nullopt);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = (packed ? pimhip_input_projection_packed : pimhip_input_projection)(out.data_ptr(), x->data_ptr(), w->data_ptr(),
                                                                             b ? b->data_ptr() : nullptr, T, K, n_out, stream);
    Py_END_ALLOW_THREADS
    return rc == PIMHIP_OK ? THPVariable_Wrap(std::move(out)) : status(rc);
}

// lstm_key(params): (addresses, version counters) of the tensors as two bytes objects, or None
PyObject* lstmKey(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    if (n != 1 || !PyList_Check(args[0])) return none();
    const Py_ssize_t count = PyList_GET_SIZE(args[0]);
    constexpr Py_ssize_t kMost = 256;
    if (count > kMost) return none();
    const void* address[kMost];
    uint32_t version[kMost];
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject* o = PyList_GET_ITEM(args[0], i);
        if (!THPVariable_Check(o)) return none();
        const at::Tensor& t = THPVariable_Unpack(o);
        if (!t.defined() || t.is_inference()) return none();
        address[i] = t.data_ptr();
        version[i] = t._version();
    }
    PyObject* a = PyBytes_FromStringAndSize(reinterpret_cast<const char*>(address), count * (Py_ssize_t)sizeof(address[0]));
    PyObject* v = PyBytes_FromStringAndSize(reinterpret_cast<const char*>(version), count * (Py_ssize_t)sizeof(version[0]));
    if (!a || !v) {
        Py_XDECREF(a);
        Py_XDECREF(v);
        return nullptr;
    }
    PyObject* both = PyTuple_Pack(2, a, v);
    Py_DECREF(a);
    Py_DECREF(v);
    return both;
}

// lstm(plan handle, input [T, 1, I] or [1, T, I], h0, c0, input size, layers * directions, hidden, directions, batch_first,
// stream): (output, hn, cn) shaped as at::lstm's
PyObject* lstm(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    const at::Tensor *x, *h0, *c0;
    void* stream;
    if (n != 10 || !tensorOf(args[1], x) || !tensorOf(args[2], h0) || !tensorOf(args[3], c0) || !streamOf(args[9], stream)) return none();
    PimHipLstmPlan* plan = static_cast<PimHipLstmPlan*>(PyLong_AsVoidPtr(args[0]));
    int64_t I, LD, H, D;
    if (!intOf(args[4], I) || !intOf(args[5], LD) || !intOf(args[6], H) || !intOf(args[7], D)) return none();
    const bool batch_first = PyObject_IsTrue(args[8]) == 1;
    if (!plan || x->dim() != 3 || x->size(batch_first ? 0 : 1) != 1 || x->size(2) != I || h0->numel() != LD * H || c0->numel() != LD * H ||
        !x->is_contiguous() || !h0->is_contiguous() || !c0->is_contiguous())
        return none();
    const int64_t T = x->size(batch_first ? 1 : 0);
    if (T < 1) return none();
    at::Tensor y = newHalf(batch_first ? at::IntArrayRef({1, T, D * H}) : at::IntArrayRef({T, 1, D * H}), *x);
    at::Tensor hn = newHalf({LD, 1, H}, *x), cn = newHalf({LD, 1, H}, *x);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = pimhip_lstm_forward(plan, x->data_ptr(), h0->data_ptr(), c0->data_ptr(), y.data_ptr(), hn.data_ptr(), cn.data_ptr(), T, stream);
    Py_END_ALLOW_THREADS
    if (rc != PIMHIP_OK) return status(rc);
    PyObject* out = PyTuple_New(3);
    if (!out) return nullptr;
    PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(y)));
    PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(hn)));
    PyTuple_SET_ITEM(out, 2, THPVariable_Wrap(std::move(cn)));
    return out;
}

// ---- bound steps: the buffers of a one-launch step, fixed once, and the call that issues it ---------------------------------
constexpr const char* kBoundStep = "pimaicompiler_amd.bound_step";
struct BoundStep {
    virtual ~BoundStep() = default;
    virtual int issue(void* stream) const = 0;
};

PyObject* capsule(BoundStep* s)
{
    PyObject* c = PyCapsule_New(s, kBoundStep, [](PyObject* o) { delete static_cast<BoundStep*>(PyCapsule_GetPointer(o, kBoundStep)); });
    if (!c) delete s;
    return c;
}

void* pointerOf(PyObject* o) { return o == Py_None ? nullptr : PyLong_AsVoidPtr(o); }

struct MoeStep : BoundStep {
    PimHipMoePlan* plan;
    const void* x;
    void *y, *logits;
    int* expert;
    int issue(void* stream) const override { return pimhip_moe_ffn_step(plan, x, y, logits, expert, stream); }
};

struct RnntStep : BoundStep {
    PimHipRnntPlan* plan;
    void* p[8];
    int run_prediction;
    int issue(void* stream) const override { return pimhip_rnnt_step(plan, p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], run_prediction, stream); }
};

struct DecoderStep : BoundStep {
    PimHipDecoderPlan* plan;
    const void *x, *att, *ctx;
    std::vector<const void*> h_prev, c_prev;
    std::vector<void*> hn, cn, outs, ctx_outs;
    void* logits;
    int issue(void* stream) const override
    {
        return pimhip_decoder_step(plan, x, att, ctx, h_prev.data(), c_prev.data(), hn.data(), cn.data(), outs.data(),
                                   ctx_outs.empty() ? nullptr : ctx_outs.data(), (int)ctx_outs.size(), logits, stream);
    }
};

// bind_moe(handle, x, y, logits, expert), bind_rnnt(handle, eight buffers, run_prediction): addresses as integers or None
PyObject* bindMoe(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    if (n != 5) return none();
    auto* s = new MoeStep();
    s->plan = static_cast<PimHipMoePlan*>(pointerOf(args[0]));
    s->x = pointerOf(args[1]);
    s->y = pointerOf(args[2]);
    s->logits = pointerOf(args[3]);
    s->expert = static_cast<int*>(pointerOf(args[4]));
    return capsule(s);
}

PyObject* bindRnnt(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    if (n != 10) return none();
    auto* s = new RnntStep();
    s->plan = static_cast<PimHipRnntPlan*>(pointerOf(args[0]));
    for (int i = 0; i < 8; ++i) s->p[i] = pointerOf(args[1 + i]);
    s->run_prediction = PyObject_IsTrue(args[9]) == 1;
    return capsule(s);
}

// bind_decoder(handle, x, att, ctx, h_prev, c_prev, hn, cn, outs, ctx_outs, logits): lists of addresses for the six in the middle
PyObject* bindDecoder(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    if (n != 11) return none();
    for (int i = 4; i < 10; ++i)
        if (!PyList_Check(args[i])) return none();
    auto* s = new DecoderStep();
    s->plan = static_cast<PimHipDecoderPlan*>(pointerOf(args[0]));
    s->x = pointerOf(args[1]);
    s->att = pointerOf(args[2]);
    s->ctx = pointerOf(args[3]);
    auto list = [](PyObject* l, auto& v) {
        for (Py_ssize_t i = 0; i < PyList_GET_SIZE(l); ++i) v.push_back(pointerOf(PyList_GET_ITEM(l, i)));
    };
    list(args[4], s->h_prev);
    list(args[5], s->c_prev);
    list(args[6], s->hn);
    list(args[7], s->cn);
    list(args[8], s->outs);
    list(args[9], s->ctx_outs);
    s->logits = pointerOf(args[10]);
    return capsule(s);
}

// issue(bound step, stream): the C ABI's status
PyObject* issue(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    void* stream;
    if (n != 2 || !streamOf(args[1], stream)) return none();
    auto* s = static_cast<BoundStep*>(PyCapsule_GetPointer(args[0], kBoundStep));
    if (!s) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = s->issue(stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

// A C++ exception (an allocation that fails) becomes a Python one.
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    return F(self, args, n);
    END_HANDLE_TH_ERRORS
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyMethodDef method(const char* name)
{
    return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<F>)), METH_FASTCALL, nullptr};
}
}  // namespace

void addFastcalls(PyObject* module)
{
    static PyMethodDef methods[] = {method<addmm>("fast_addmm"),           method<matmul>("fast_matmul"),
                                    method<linear>("fast_linear"),         method<group>("fast_group"),
                                    method<projection>("fast_projection"), method<lstmKey>("lstm_key"),
                                    method<lstm>("fast_lstm"),             method<bindMoe>("bind_moe"),
                                    method<bindRnnt>("bind_rnnt"),         method<bindDecoder>("bind_decoder"),
                                    method<issue>("issue"),                {nullptr, nullptr, 0, nullptr}};
    if (PyModule_AddFunctions(module, methods) != 0) throw pybind11::error_already_set();
}
