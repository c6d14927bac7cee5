// The call path of nanoinfer_amd.quant in native code: one C call per operation that
// checks its tensors, takes the outputs and the workspace from torch's allocator and
// launches on the current stream. The same work in Python and ctypes (attribute reads,
// two torch.empty, an 18-argument foreign call) took 7 us of every call, more than
// most decode kernels: m = 1, n = 4864, k = 896 int8 10.9 -> 4.3 us a call, W8A8 m = 16, n =
// 8960, k = 1536 15.0 -> 8.8; a W8A8 decoder layer over 24 tokens 151 -> 76.
//
// Each function handles the plain case (contiguous tensors of the expected types and
// shapes on the current device) and returns None otherwise, or when the library or the
// allocator reports an error: the caller then runs its Python path, which converts what
// it accepts and raises what it refuses.
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "../../../include/nq.h"

namespace {

// A borrowed view of a plain device tensor.
struct In {
    const at::Tensor* t = nullptr;
    bool plain(PyObject* o, int device) {
        if (!THPVariable_CheckExact(o)) return false;
        t = &THPVariable_Unpack(o);
        return t->is_cuda() && t->layout() == c10::kStrided && t->has_storage() && t->get_device() == device &&
               !t->is_neg() && !t->is_conj() && !t->unsafeGetTensorImpl()->is_python_dispatch();
    }
    bool packed(PyObject* o, int device) { return plain(o, device) && t->is_contiguous(); }
    bool act() const { return t->scalar_type() == at::kFloat || t->scalar_type() == at::kHalf; }
    nq_dtype dt() const { return t->scalar_type() == at::kFloat ? NQ_F32 : NQ_F16; }
    void* p() const { return t->data_ptr(); }
    int64_t size(int i) const { return t->size(i); }
};

at::Tensor empty(at::IntArrayRef shape, at::ScalarType st, int device) {
    return at::empty(shape, at::TensorOptions().dtype(st).device(at::kCUDA, static_cast<c10::DeviceIndex>(device)));
}

// None or an fp32 vector of `n`.
bool bias_ok(PyObject* o, int device, int64_t n, const float** out) {
    *out = nullptr;
    if (o == Py_None) return true;
    In b;
    if (!b.packed(o, device) || b.t->scalar_type() != at::kFloat || b.t->numel() != n) return false;
    *out = static_cast<const float*>(b.p());
    return true;
}

// torch.float32 / torch.float16, or None for `none`.
bool out_type(PyObject* o, at::ScalarType none, at::ScalarType* st) {
    *st = o == Py_None ? none : THPDtype_Check(o) ? reinterpret_cast<THPDtype*>(o)->scalar_type : at::kByte;
    return *st == at::kFloat || *st == at::kHalf;
}

nq_dtype code(at::ScalarType st) { return st == at::kFloat ? NQ_F32 : NQ_F16; }

int64_t integer(PyObject* o) { return PyLong_AsLongLong(o); }

// Runs f(device, stream) -> the result or an undefined tensor; no exception leaves.
template <int N, typename F>
PyObject* call(Py_ssize_t n, F f) {
    if (n != N) {
        PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
        return nullptr;
    }
    PyObject* r = nullptr;
    try {
        const int device = c10::hip::current_device();
        r = f(device, c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(device)).stream());
    } catch (...) {
        r = nullptr;
    }
    if (PyErr_Occurred()) PyErr_Clear();
    if (r) return r;
    Py_RETURN_NONE;
}

// The library call without the interpreter lock, as ctypes makes it. What f throws (a
// tensor that gives no data pointer) finds the lock held again.
struct Unlocked {
    PyThreadState* const state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};
template <typename F>
bool launch(F f) {
    const Unlocked unlocked;
    return f() == NQ_OK;
}

PyObject* wrap(at::Tensor t) { return THPVariable_Wrap(std::move(t)); }
PyObject* tuple(std::initializer_list<at::Tensor> ts) {
    PyObject* r = PyTuple_New(static_cast<Py_ssize_t>(ts.size()));
    Py_ssize_t i = 0;
    for (const at::Tensor& t : ts) PyTuple_SET_ITEM(r, i++, THPVariable_Wrap(t));
    return r;
}

// linear(kind, x, q, scale, bias, out_dtype, out, in, group, path); kind 0 q8, 1 q4g, 2 w8a8
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return call<10>(n, [&](int dev, hipStream_t s) -> PyObject* {
        const int64_t kind = integer(a[0]), out = integer(a[6]), in = integer(a[7]), group = integer(a[8]);
        const int path = static_cast<int>(integer(a[9]));
        In x, q, sc;
        const float* b;
        at::ScalarType yt;
        if (!x.packed(a[1], dev) || x.t->dim() != 2 || x.size(1) != in || !x.act() || !q.plain(a[2], dev) ||
            !sc.plain(a[3], dev) || !bias_ok(a[4], dev, out, &b) || !out_type(a[5], x.t->scalar_type(), &yt) || out < 0 || in < 0)
            return nullptr;
        const int64_t m = x.size(0);
        if (kind == 1) {
            if (group <= 0 || q.t->numel() != out * ((in + 1) / 2) || sc.t->numel() != out * ((in + group - 1) / group) || !sc.act())
                return nullptr;
        } else if (q.t->numel() != out * in || sc.t->numel() != out || sc.t->scalar_type() != at::kFloat) {
            return nullptr;
        }
        const at::Tensor y = empty({m, out}, yt, dev);
        const size_t need = kind == 2 ? nq_linear_w8a8_workspace_preferred(m, out, in) : nq_linear_wq_workspace_preferred(m, out, in);
        at::Tensor ws;
        if (need || kind == 2) ws = empty({static_cast<int64_t>(need < 256 ? 256 : need)}, at::kByte, dev);
        void* wp = ws.defined() ? ws.data_ptr() : nullptr;
        void* yp = y.data_ptr();
        const bool ok = launch([&] {
            if (kind == 0)
                return nq_linear_q8_ex(x.p(), x.dt(), static_cast<const int8_t*>(q.p()), static_cast<const float*>(sc.p()), b, yp,
                                       code(yt), m, out, in, wp, need, path, s);
            if (kind == 1)
                return nq_linear_q4g_ex(x.p(), x.dt(), static_cast<const uint8_t*>(q.p()), sc.p(), sc.dt(), group, b, yp, code(yt), m,
                                        out, in, wp, need, path, s);
            return nq_linear_w8a8(x.p(), x.dt(), static_cast<const int8_t*>(q.p()), static_cast<const float*>(sc.p()), b, yp, code(yt),
                                  m, out, in, wp, static_cast<size_t>(ws.numel()), path, s);
        });
        return ok ? wrap(y) : nullptr;
    });
}

// gemm_w8a8(xq, a_scale, q, scale, bias, out_dtype, out, in, path)
PyObject* gemm_w8a8(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return call<9>(n, [&](int dev, hipStream_t s) -> PyObject* {
        const int64_t out = integer(a[6]), in = integer(a[7]);
        const int path = static_cast<int>(integer(a[8]));
        In x, as, q, sc;
        const float* b;
        at::ScalarType yt;
        if (!x.packed(a[0], dev) || x.t->scalar_type() != at::kChar || x.t->dim() != 2 || x.size(1) != in || !as.packed(a[1], dev) ||
            as.t->scalar_type() != at::kFloat || as.t->numel() != x.size(0) || !q.plain(a[2], dev) || q.t->numel() != out * in ||
            !sc.plain(a[3], dev) || sc.t->numel() != out || sc.t->scalar_type() != at::kFloat || !bias_ok(a[4], dev, out, &b) ||
            a[5] == Py_None || !out_type(a[5], at::kHalf, &yt))
            return nullptr;
        const int64_t m = x.size(0);
        const at::Tensor y = empty({m, out}, yt, dev);
        const size_t need = nq_gemm_w8a8_workspace_preferred(m, out, in);
        at::Tensor ws;
        if (need) ws = empty({static_cast<int64_t>(need)}, at::kByte, dev);
        void *wp = need ? ws.data_ptr() : nullptr, *yp = y.data_ptr();
        const bool ok = launch([&] {
            return nq_gemm_w8a8(static_cast<const int8_t*>(x.p()), static_cast<const float*>(as.p()), static_cast<const int8_t*>(q.p()),
                                static_cast<const float*>(sc.p()), b, yp, code(yt), m, out, in, wp, need, path, s);
        });
        return ok ? wrap(y) : nullptr;
    });
}

// act_quant(x) -> (xq, scale)
PyObject* act_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return call<1>(n, [&](int dev, hipStream_t s) -> PyObject* {
        In x;
        if (!x.packed(a[0], dev) || x.t->dim() != 2 || !x.act()) return nullptr;
        const int64_t m = x.size(0), k = x.size(1);
        const at::Tensor xq = empty({m, k}, at::kChar, dev), sc = empty({m}, at::kFloat, dev);
        const bool ok = launch([&] {
            return nq_act_quant_i8(x.p(), x.dt(), m, k, xq.data_ptr<int8_t>(), sc.data_ptr<float>(), s);
        });
        return ok ? tuple({xq, sc}) : nullptr;
    });
}

// act_quant_heads(a [heads, s, d]) -> (xq [s, heads * d], scale)
PyObject* act_quant_heads(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return call<1>(n, [&](int dev, hipStream_t s) -> PyObject* {
        In x;
        if (!x.packed(a[0], dev) || x.t->dim() != 3 || !x.act()) return nullptr;
        const int64_t h = x.size(0), rows = x.size(1), d = x.size(2);
        const at::Tensor xq = empty({rows, h * d}, at::kChar, dev), sc = empty({rows}, at::kFloat, dev);
        const bool ok = launch([&] {
            return nq_act_quant_i8_heads(x.p(), x.dt(), h, rows, d, xq.data_ptr<int8_t>(), sc.data_ptr<float>(), s);
        });
        return ok ? tuple({xq, sc}) : nullptr;
    });
}

bool norm_weight(PyObject* o, int dev, int64_t k, In* w) {
    return w->packed(o, dev) && w->t->scalar_type() == at::kFloat && w->t->numel() == k;
}

// rmsnorm_quant(x, w, eps) -> (xq, scale)
PyObject* rmsnorm_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return call<3>(n, [&](int dev, hipStream_t s) -> PyObject* {
        In x, w;
        if (!x.packed(a[0], dev) || x.t->dim() != 2 || !x.act() || !norm_weight(a[1], dev, x.size(1), &w) || !PyFloat_Check(a[2]))
            return nullptr;
        const int64_t m = x.size(0), k = x.size(1);
        const float eps = static_cast<float>(PyFloat_AS_DOUBLE(a[2]));
        const at::Tensor xq = empty({m, k}, at::kChar, dev), sc = empty({m}, at::kFloat, dev);
        const bool ok = launch([&] {
            return nq_rmsnorm_quant_i8(x.p(), x.dt(), static_cast<const float*>(w.p()), eps, m, k, xq.data_ptr<int8_t>(),
                                       sc.data_ptr<float>(), s);
        });
        return ok ? tuple({xq, sc}) : nullptr;
    });
}

// add_rmsnorm_quant(x, r, w, eps) -> (h, xq, scale)
PyObject* add_rmsnorm_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return call<4>(n, [&](int dev, hipStream_t s) -> PyObject* {
        In x, r, w;
        if (!x.packed(a[0], dev) || x.t->dim() != 2 || !x.act() || !r.packed(a[1], dev) || r.t->sizes() != x.t->sizes() ||
            r.t->scalar_type() != x.t->scalar_type() || !norm_weight(a[2], dev, x.size(1), &w) || !PyFloat_Check(a[3]))
            return nullptr;
        const int64_t m = x.size(0), k = x.size(1);
        const float eps = static_cast<float>(PyFloat_AS_DOUBLE(a[3]));
        const at::Tensor h = empty({m, k}, x.t->scalar_type(), dev), xq = empty({m, k}, at::kChar, dev), sc = empty({m}, at::kFloat, dev);
        const bool ok = launch([&] {
            return nq_add_rmsnorm_quant_i8(x.p(), r.p(), x.dt(), static_cast<const float*>(w.p()), eps, m, k, h.data_ptr(),
                                           xq.data_ptr<int8_t>(), sc.data_ptr<float>(), s);
        });
        return ok ? tuple({h, xq, sc}) : nullptr;
    });
}

// silu_mul_quant(gate, up) -> (xq, scale); silu_mul_quant of the halves of one [m, 2 i] tensor when up is None
PyObject* silu_mul_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return call<2>(n, [&](int dev, hipStream_t s) -> PyObject* {
        In g, u;
        if (!g.plain(a[0], dev) || g.t->dim() != 2 || !g.act() || g.t->stride(1) != 1) return nullptr;
        int64_t m = g.size(0), k = g.size(1);
        const char* up;
        if (a[1] == Py_None) {
            if (k % 2) return nullptr;
            k /= 2;
            up = static_cast<const char*>(g.p()) + k * g.t->element_size();
        } else {
            if (!u.plain(a[1], dev) || u.t->sizes() != g.t->sizes() || u.t->strides() != g.t->strides() ||
                u.t->scalar_type() != g.t->scalar_type())
                return nullptr;
            up = static_cast<const char*>(u.p());
        }
        const at::Tensor xq = empty({m, k}, at::kChar, dev), sc = empty({m}, at::kFloat, dev);
        const bool ok = launch([&] {
            return nq_silu_mul_quant_i8(g.p(), up, g.dt(), m, k, g.t->stride(0), xq.data_ptr<int8_t>(), sc.data_ptr<float>(), s);
        });
        return ok ? tuple({xq, sc}) : nullptr;
    });
}

// rope_qkv(qkv, heads, kv_heads, head_dim, cos, sin) -> (q, k, v) head-major
PyObject* rope_qkv(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return call<6>(n, [&](int dev, hipStream_t s) -> PyObject* {
        In x, c, sn;
        const int64_t h = integer(a[1]), kv = integer(a[2]), d = integer(a[3]);
        if (!x.plain(a[0], dev) || x.t->dim() != 2 || !x.act() || x.t->stride(1) != 1 || h < 0 || kv < 0 || d < 0 ||
            !c.packed(a[4], dev) || !sn.packed(a[5], dev) || c.t->scalar_type() != at::kFloat || sn.t->scalar_type() != at::kFloat ||
            c.t->dim() != 2 || c.t->sizes() != sn.t->sizes() || c.size(1) != d || c.size(0) < x.size(0))
            return nullptr;
        const int64_t rows = x.size(0);
        const at::ScalarType st = x.t->scalar_type();
        const at::Tensor q = empty({h, rows, d}, st, dev), k = empty({kv, rows, d}, st, dev), v = empty({kv, rows, d}, st, dev);
        const bool ok = launch([&] {
            return nq_rope_qkv(x.p(), x.dt(), rows, x.t->stride(0), h, kv, d, static_cast<const float*>(c.p()),
                               static_cast<const float*>(sn.p()), q.data_ptr(), k.data_ptr(), v.data_ptr(), s);
        });
        return ok ? tuple({q, k, v}) : nullptr;
    });
}

// Whether something besides the kernel wants to see or steer a torch call: a tracer, a
// dispatch or torch-function mode, autocast, or a selection among torch's own attentions.
bool torch_call_observed() {
    const at::Context& c = at::globalContext();
    return torch::jit::tracer::isTracing() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
           at::impl::torch_function_mode_enabled() || at::autocast::is_autocast_enabled(at::kCUDA) ||
           !(c.userEnabledFlashSDP() && c.userEnabledMemEfficientSDP() && c.userEnabledMathSDP());
}

// attention(q [heads, s, d], k, v [kv, s, d]) -> [heads, s, d], causal, fp16 heads of 64 or
// 128. It stands where a differentiable torch call stands otherwise, so it declines
// whatever autograd or forward mode follows, and every call that torch_call_observed.
PyObject* attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return call<3>(n, [&](int dev, hipStream_t s) -> PyObject* {
        In q, k, v;
        if (torch_call_observed() || !q.packed(a[0], dev) || !k.packed(a[1], dev) || !v.packed(a[2], dev))
            return nullptr;
        for (const In* t : {&q, &k, &v})
            if (t->t->dim() != 3 || t->t->scalar_type() != at::kHalf || t->t->unsafeGetTensorImpl()->autograd_meta() != nullptr)
                return nullptr;
        const int64_t h = q.size(0), rows = q.size(1), d = q.size(2), kv = k.size(0);
        if ((d != 64 && d != 128) || k.t->sizes() != v.t->sizes() || k.size(1) != rows || k.size(2) != d || kv < 1 || h < 1 || h % kv)
            return nullptr;
        // Longer rows are torch's, unmeasured, and so are many heads of long ones: 16 queries to each
        // read of K and V bound this kernel once its workgroups fill the GPU (us, this / torch: 28 heads
        // of 128, 768 tokens 40 / 44, 1024 64 / 55; 16 heads, 1536 73 / 84, 2048 112 / 104; 64 heads, 512
        // 46 / 40; heads of 64: 32, 768 tokens 30 / 31, 1024 45 / 38).
        if (rows > (d == 64 ? 1024 : 2048) || h * rows > 24576) return nullptr;
        const at::Tensor out = empty({h, rows, d}, at::kHalf, dev);
        const bool ok = launch([&] { return nq_attention_causal_f16(q.p(), k.p(), v.p(), h, kv, rows, d, out.data_ptr(), s); });
        return ok ? wrap(out) : nullptr;
    });
}

// quantize(w, group, scale_dtype) -> (codes, scales); group 0: int8 per row
PyObject* quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return call<3>(n, [&](int dev, hipStream_t s) -> PyObject* {
        In w;
        const int64_t group = integer(a[1]);
        at::ScalarType st;
        if (!w.packed(a[0], dev) || w.t->dim() != 2 || w.t->scalar_type() != at::kFloat || group < 0 || !out_type(a[2], at::kFloat, &st))
            return nullptr;
        const int64_t out = w.size(0), k = w.size(1);
        const float* wp = static_cast<const float*>(w.p());
        const at::Tensor q = group ? empty({out, (k + 1) / 2}, at::kByte, dev) : empty({out, k}, at::kChar, dev);
        const at::Tensor sc = group ? empty({out, (k + group - 1) / group}, st, dev) : empty({out}, at::kFloat, dev);
        const bool ok = launch([&] {
            if (group) return nq_quantize_q4g(wp, out, k, group, q.data_ptr<uint8_t>(), sc.data_ptr(), code(st), s);
            return nq_quantize_q8(wp, out, k, q.data_ptr<int8_t>(), sc.data_ptr<float>(), s);
        });
        return ok ? tuple({q, sc}) : nullptr;
    });
}

#define NQ_CALL(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {NQ_CALL(linear), NQ_CALL(gemm_w8a8), NQ_CALL(act_quant), NQ_CALL(act_quant_heads), NQ_CALL(rmsnorm_quant),
                         NQ_CALL(add_rmsnorm_quant), NQ_CALL(silu_mul_quant), NQ_CALL(rope_qkv), NQ_CALL(attention), NQ_CALL(quantize),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", "Native call path of nanoinfer_amd.quant.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() { return PyModule_Create(&module); }
