// CPython extension in front of the C ABI: the eager call path of the ops and of the fp8 linear layers.
//
// What bounds a small eager call is the host.  Checking tensors, asking torch for the stream and the
// output, carving arguments and going through ctypes took 23 us per linear in Python where its one kernel
// takes 4 - 6 us on the GPU (an MLP 34 us, a decoder layer 170 us); here the same steps are a few hundred
// nanoseconds plus the launch itself.
//
// Every function either does the whole call and returns its result, or returns None having launched
// nothing: the Python op then takes its own path, which checks the arguments one by one, handles the forms
// this file leaves alone (copies of unaligned rows, empty inputs, another current device) and raises the
// error a caller sees.  Nothing about results lives here: the kernels, their choice and the workspace
// (phyai_amd.ops._workspaces, or the owner in scope while a graph is recorded) are those of the Python path.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <dlfcn.h>

#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/phyai_fp8.h"
#include "host_entry.h"

namespace {

// ---- what bind() was given -----------------------------------------------------------------------------
struct Lib {
    decltype(&phyai_fp8_linear) linear;
    decltype(&phyai_fp8_linear_addcmul) linear_addcmul;
    decltype(&phyai_fp8_gemm) gemm;
    decltype(&phyai_fp8_gemm_addcmul) gemm_addcmul;
    decltype(&phyai_fp8_mlp) mlp;
    decltype(&phyai_fp8_adarmsnorm_linear) norm_linear;
    decltype(&phyai_fp8_adarmsnorm_mlp) norm_mlp;
    decltype(&phyai_fp8_linear_workspace_bytes) linear_ws;
    decltype(&phyai_fp8_mlp_workspace_bytes) mlp_ws;
    decltype(&phyai_fp8_quant_rowwise) quant_rowwise;
    decltype(&phyai_fp8_weight_quant_rowwise) weight_quant;
    decltype(&phyai_fp8_weight_to_operand_order) relay;
    decltype(&phyai_fp8_weight_to_operand_order_inplace) relay_inplace;
    decltype(&phyai_host_relay_gated) relay_gated;
    decltype(&phyai_fp8_linear_per_tensor) per_tensor;
    decltype(&phyai_fp8_rmsnorm_quant) rmsnorm;
    decltype(&phyai_fp8_adarmsnorm_quant) adarmsnorm;
} lib = {};

struct Py {
    PyObject *workspaces, *owner, *reserve, *epilogues, *layouts, *view_type, *per_channel, *per_tensor;
} py = {};
struct PyLayers {
    PyObject *dispatch_dict, *mode, *kernel_type, *kernel_apply, *quantize_activation;
} pl = {};
// what the calls of modules need: phyai_amd.ops's dictionary, this extension, nn.Module and its __call__, the tables of
// hooks that apply to every module, and the forward methods that the calls below stand for
struct PyModules {
    PyObject *ops_dict, *self, *module_type, *module_call, *global_hooks, *linear_forward, *mlp_forward, *linear_forward_fused,
        *linear_forward_addcmul, *norm_forward_fp8, *linear_supports, *linear_call;
} pm = {};

PyObject *s_dispatcher, *s_generation, *s_selected, *s_params_dtype, *s_skip_bias_add, *s_bias;
PyObject *s_host, *s_call, *s_forward, *s_forward_fused, *s_forward_addcmul, *s_forward_fp8, *s_supports, *s_fuse_activation, *s_gated,
    *s_epilogue, *s_modules, *s_gate_up, *s_down, *s_fc1, *s_fc2, *s_residual, *s_gate, *s_compiled, *s_hooks[4];
PyObject *s_parameters, *s_weight, *s_weight_scale, *s_input_scale, *s_stream_weights, *s_weight_layout,
    *s_spec, *s_granularity, *s_apply, *s_quantize;

PyObject* declined() {
    PyErr_Clear();
    Py_RETURN_NONE;
}

// ---- tensors ---------------------------------------------------------------------------------------------
const at::Tensor* tensor(PyObject* o) { return o && THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }
PyObject* none_if_null(PyObject* o) { return o ? o : Py_None; }

struct Rows {
    const void* p;
    int64_t M, K, ld;
};
// The [M, K] view of a tensor whose rows the kernels can read as they lie.
bool rows_of(const at::Tensor& t, at::ScalarType dtype, Rows* r) {
    if (!t.is_cuda() || t.scalar_type() != dtype || t.dim() < 1 || t.numel() == 0) return false;
    const int64_t d = t.dim();
    r->K = t.size(d - 1);
    r->M = t.numel() / r->K;
    if (t.stride(d - 1) != 1) return false;
    if (t.is_contiguous()) r->ld = r->K;
    else if (d == 2) r->ld = r->M > 1 ? t.stride(0) : r->K;
    else return false;
    r->p = t.const_data_ptr();
    return r->ld >= r->K && r->ld % 8 == 0 && (reinterpret_cast<uintptr_t>(r->p) & 15) == 0;
}
bool codes_dtype(const at::Tensor& t) {
    return t.scalar_type() == at::kFloat8_e4m3fn || t.scalar_type() == at::kByte;
}
bool vector_of(const at::Tensor* t, at::ScalarType dtype, int64_t n) {
    return t && t->is_cuda() && t->scalar_type() == dtype && t->numel() == n && t->is_contiguous();
}

// The device a call runs on and the stream of it; calls for another device than the current one are left
// to the Python path.
struct Where {
    at::Device dev{at::kCUDA, 0};
    hipStream_t stream = nullptr;
};
bool where(const at::Tensor& x, Where* w) {
    const auto cur = c10::hip::current_device();
    if (x.device().index() != cur) return false;
    w->dev = x.device();
    w->stream = c10::hip::getCurrentHIPStream(cur).stream();
    return true;
}

// Fresh tensor shaped like `lead` with its last dimension replaced.
at::Tensor fresh(const at::Tensor& lead, int64_t last, at::ScalarType dtype, const at::Device& dev) {
    c10::SmallVector<int64_t, 6> shape(lead.sizes().begin(), lead.sizes().end());
    shape.back() = last;
    return at::Tensor(at::detail::empty_cuda(shape, dtype, dev, std::nullopt));
}
bool shaped(const at::Tensor* t, const at::Tensor& lead, int64_t last, at::ScalarType dtype) {
    if (!t || !t->is_cuda() || t->scalar_type() != dtype || t->dim() != lead.dim() || !t->is_contiguous()) return false;
    for (int64_t i = 0; i + 1 < lead.dim(); ++i)
        if (t->size(i) != lead.size(i)) return false;
    return t->size(lead.dim() - 1) == last;
}

// ---- workspace -----------------------------------------------------------------------------------------------
struct Scratch {
    void* p;
    size_t n;
};
bool workspace(size_t need, const Where& w, Scratch* s) {
    PyObject* owner = nullptr;
    if (PyContextVar_Get(py.owner, nullptr, &owner) < 0) return false;
    const bool shared = owner == nullptr || owner == Py_None;
    Py_XDECREF(owner);
    if (shared) {
        PyObject* key = Py_BuildValue("iK", (int)w.dev.index(), (unsigned long long)reinterpret_cast<uintptr_t>(w.stream));
        if (!key) return false;
        const at::Tensor* t = tensor(PyDict_GetItemWithError(py.workspaces, key));
        Py_DECREF(key);
        if (t && (size_t)t->numel() >= need) {
            *s = {t->mutable_data_ptr(), (size_t)t->numel()};
            return true;
        }
    }
    PyObject* o = PyObject_CallFunction(py.reserve, "K", (unsigned long long)need);
    const at::Tensor* t = tensor(o);
    if (t) *s = {t->mutable_data_ptr(), (size_t)t->numel()};
    const bool ok = t != nullptr;
    Py_XDECREF(o);   // its owner or the table of workspaces keeps it
    return ok;
}

// ---- one linear -------------------------------------------------------------------------------------------------
bool is_gated(int epi) { return epi >= PHYAI_FP8_EPI_GEGLU_TANH && epi <= PHYAI_FP8_EPI_SWIGLU; }

// Epilogue (name, number or None) and the flag bits of the weight.
bool epilogue_of(PyObject* o, int* epi) {
    if (o == Py_None) { *epi = 0; return true; }
    if (PyLong_CheckExact(o)) {
        *epi = (int)PyLong_AsLong(o);
        return *epi >= 0 && *epi <= PHYAI_FP8_EPI_GELU_ERF;
    }
    PyObject* v = PyDict_GetItemWithError(py.epilogues, o);
    if (!v) return false;
    *epi = (int)PyLong_AsLong(v);
    return true;
}
bool flags_of(PyObject* layout, bool stream, int epi, int* flags) {
    int f = 0;
    if (layout != Py_None) {
        PyObject* v = PyDict_GetItemWithError(py.layouts, layout);
        if (!v) return false;
        f = (int)PyLong_AsLong(v);
        if (f && (f == PHYAI_FP8_FLAG_W_OPERAND_GATED) != is_gated(epi)) return false;
    }
    *flags = f | (stream ? PHYAI_FP8_FLAG_STREAM_WEIGHTS : 0);
    return true;
}

struct Weight {
    const void* w;
    const float* scale;
    const void* bias;
    int64_t N;
};
bool weight_of(PyObject* w_, PyObject* s_, PyObject* b_, int64_t K, Weight* out) {
    const at::Tensor *w = tensor(w_), *s = tensor(s_), *b = tensor(b_);
    if (!w || !s || (b_ != Py_None && !b)) return false;
    if (!w->is_cuda() || w->dim() != 2 || !codes_dtype(*w) || !w->is_contiguous() || w->size(1) != K) return false;
    const int64_t N = w->size(0);
    if (N == 0 || K % 16 != 0 || N % 16 != 0 || !vector_of(s, at::kFloat, N)) return false;
    if (b && !vector_of(b, at::kBFloat16, N)) return false;
    *out = {w->const_data_ptr(), s->const_data_ptr<float>(), b ? b->const_data_ptr() : nullptr, N};
    return true;
}

struct Residual {
    const void *residual, *gate;
    int64_t ld_gate, gate_rows;
};
bool residual_of(PyObject* r_, PyObject* g_, const at::Tensor& x, int64_t M, int64_t N, int epi, Residual* out) {
    *out = {nullptr, nullptr, 0, 0};
    if (r_ == Py_None && g_ == Py_None) return true;
    const at::Tensor *r = tensor(r_), *g = tensor(g_);
    if (!r || !g || epi != 0 || !shaped(r, x, N, at::kBFloat16)) return false;
    if (!g->is_cuda() || g->scalar_type() != at::kBFloat16 || g->dim() < 1 || g->size(g->dim() - 1) != N || g->numel() == 0) return false;
    const int64_t rows = g->numel() / N;
    if (!g->is_contiguous() || M % rows != 0) return false;
    *out = {r->const_data_ptr(), g->const_data_ptr(), N, rows};
    return true;
}

// Rows of scale | shift | gate of an adaptive norm of width D.
struct Modulation {
    const uint8_t* p;
    int64_t rows, ld, D;
    double eps;
};
bool modulation_of(PyObject* m_, PyObject* eps, int64_t D, int64_t M, Modulation* out) {
    const at::Tensor* m = tensor(m_);
    Rows q;
    if (!m || m->dim() != 2 || !rows_of(*m, at::kBFloat16, &q) || q.K != 3 * D || D % 8 != 0 || M % q.M != 0) return false;
    *out = {static_cast<const uint8_t*>(q.p), q.M, q.M > 1 ? q.ld : q.K, D, eps ? PyFloat_AsDouble(eps) : 0.0};
    return !PyErr_Occurred();
}
// residual + gate part of a modulation row (one row per group of token rows)
bool residual_gated_by(PyObject* r_, PyObject* m_, const at::Tensor& x, int64_t M, int64_t N, Residual* out) {
    const at::Tensor* r = tensor(r_);
    Modulation m;
    if (!r || !shaped(r, x, N, at::kBFloat16) || !modulation_of(m_, nullptr, N, M, &m)) return false;
    *out = {r->const_data_ptr(), m.p + 4 * N, m.ld, m.rows};
    return true;
}

// bf16 rows `x_`, or codes `x_` with their scales `xs_` when that is given -> output tensor, null when declined.
PyObject* linear_call(PyObject* x_, PyObject* xs_, PyObject* w_, PyObject* ws_, PyObject* b_, int epi, PyObject* layout,
                      bool stream, PyObject* out_, PyObject* res_, PyObject* gate_, bool gate_in_modulation = false,
                      PyObject* mod_ = nullptr, PyObject* eps_ = nullptr) {
    const at::Tensor* x = tensor(x_);
    if (!x) return nullptr;
    Rows r;
    const bool codes = xs_ != nullptr;
    if (codes ? !(codes_dtype(*x) && x->is_contiguous() && rows_of(*x, x->scalar_type(), &r)) : !rows_of(*x, at::kBFloat16, &r))
        return nullptr;
    Where at_;
    Weight w;
    int flags;
    if (!where(*x, &at_) || !weight_of(w_, ws_, b_, r.K, &w) || !flags_of(layout, stream, epi, &flags)) return nullptr;
    if (is_gated(epi) && w.N % 32 != 0) return nullptr;
    const float* xs = nullptr;
    int scalar = 0;
    if (codes) {
        const at::Tensor* s = tensor(xs_);
        if (!s || !(vector_of(s, at::kFloat, r.M) || vector_of(s, at::kFloat, 1))) return nullptr;
        xs = s->const_data_ptr<float>();
        scalar = s->numel() == 1 && r.M != 1;
    }
    Residual rg;
    if (gate_in_modulation ? epi != 0 || !residual_gated_by(res_, gate_, *x, r.M, w.N, &rg) : !residual_of(res_, gate_, *x, r.M, w.N, epi, &rg))
        return nullptr;
    Modulation mod = {};
    if (mod_ && (codes || rg.residual || !modulation_of(mod_, eps_, r.K, r.M, &mod))) return nullptr;
    const int64_t n_out = is_gated(epi) ? w.N / 2 : w.N;
    at::Tensor made;
    void* out;
    if (out_ == Py_None) {
        made = fresh(*x, n_out, at::kBFloat16, at_.dev);
        out = made.mutable_data_ptr();
    } else {
        const at::Tensor* o = tensor(out_);
        if (!shaped(o, *x, n_out, at::kBFloat16)) return nullptr;
        out = o->mutable_data_ptr();
    }
    Scratch ws;
    if (!workspace(lib.linear_ws(r.M, w.N, r.K, epi), at_, &ws)) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    if (mod_)
        rc = lib.norm_linear(r.p, r.ld, mod.p, mod.ld, mod.rows, (float)mod.eps, w.w, w.scale, w.bias, out, n_out, r.M, w.N, r.K,
                             epi | flags, ws.p, ws.n, at_.stream);
    else if (codes)
        rc = rg.residual ? lib.gemm_addcmul(r.p, xs, scalar, w.w, w.scale, w.bias, rg.residual, w.N, rg.gate, rg.ld_gate, rg.gate_rows,
                                            out, n_out, r.M, w.N, r.K, flags, ws.p, ws.n, at_.stream)
                         : lib.gemm(r.p, xs, scalar, w.w, w.scale, w.bias, out, n_out, r.M, w.N, r.K, epi | flags, ws.p, ws.n, at_.stream);
    else
        rc = rg.residual ? lib.linear_addcmul(r.p, r.ld, w.w, w.scale, w.bias, rg.residual, w.N, rg.gate, rg.ld_gate, rg.gate_rows, out,
                                              n_out, r.M, w.N, r.K, flags, ws.p, ws.n, at_.stream)
                         : lib.linear(r.p, r.ld, w.w, w.scale, w.bias, out, n_out, r.M, w.N, r.K, epi | flags, ws.p, ws.n, at_.stream);
    Py_END_ALLOW_THREADS
    if (rc != 0) return nullptr;   // the Python path meets the same status and reports it
    if (out_ != Py_None) {
        Py_INCREF(out_);
        return out_;
    }
    return THPVariable_Wrap(std::move(made));
}

// bf16 rows, one static scale for all of them
PyObject* linear_static_call(PyObject* x_, PyObject* in_scale_, PyObject* w_, PyObject* ws_, PyObject* b_, int epi,
                             PyObject* layout, bool stream, PyObject* res_, PyObject* gate_) {
    const at::Tensor *x = tensor(x_), *s = tensor(in_scale_);
    Rows r;
    Where at_;
    Weight w;
    int flags;
    Residual rg;
    if (!x || !vector_of(s, at::kFloat, 1) || !rows_of(*x, at::kBFloat16, &r) || !where(*x, &at_) || !weight_of(w_, ws_, b_, r.K, &w) ||
        !flags_of(layout, stream, epi, &flags) || (is_gated(epi) && w.N % 32 != 0) || !residual_of(res_, gate_, *x, r.M, w.N, epi, &rg))
        return nullptr;
    const int64_t n_out = is_gated(epi) ? w.N / 2 : w.N;
    at::Tensor made = fresh(*x, n_out, at::kBFloat16, at_.dev);
    Scratch ws;
    if (!workspace(lib.linear_ws(r.M, w.N, r.K, epi), at_, &ws)) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = lib.per_tensor(r.p, r.ld, s->const_data_ptr<float>(), w.w, w.scale, w.bias, rg.residual, w.N, rg.gate, rg.ld_gate, rg.gate_rows,
                        made.mutable_data_ptr(), n_out, r.M, w.N, r.K, epi | flags, ws.p, ws.n, at_.stream);
    Py_END_ALLOW_THREADS
    return rc == 0 ? THPVariable_Wrap(std::move(made)) : nullptr;
}

// linear(x, weight, weight_scale, bias, epilogue, out, residual, gate, stream_weights, weight_layout)
PyObject* py_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS   // e.g. torch out of memory
    int epi;
    if (n != 10 || !epilogue_of(a[4], &epi)) return declined();
    PyObject* y = linear_call(a[0], nullptr, a[1], a[2], a[3], epi, a[9], PyObject_IsTrue(a[8]) == 1, a[5], a[6], a[7]);
    return y ? y : declined();
    END_HANDLE_TH_ERRORS
}
// gemm(xq, x_scale, weight, weight_scale, bias, epilogue, out, residual, gate, stream_weights, weight_layout)
PyObject* py_gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    int epi;
    if (n != 11 || !epilogue_of(a[5], &epi)) return declined();
    PyObject* y = linear_call(a[0], a[1], a[2], a[3], a[4], epi, a[10], PyObject_IsTrue(a[9]) == 1, a[6], a[7], a[8]);
    return y ? y : declined();
    END_HANDLE_TH_ERRORS
}

// ---- layers -------------------------------------------------------------------------------------------------------
// A reference of its own.  The dictionaries that a module's parameters are read from belong to the program: another
// thread (the GIL is released around a launch) or Python code that a call runs into (a property of the spec, the
// workspace's allocation) may put something else there before the launch has used the addresses it was given.
struct Ref {
    PyObject* p = nullptr;
    Ref() = default;
    Ref(const Ref&) = delete;
    Ref& operator=(const Ref&) = delete;
    ~Ref() { Py_XDECREF(p); }
    void set(PyObject* borrowed) {
        Py_XINCREF(borrowed);
        Py_XDECREF(p);
        p = borrowed;
    }
    operator PyObject*() const { return p; }
};

// What the HIP kernel needs of a linear layer, read from the module's own dictionaries (a module's
// __getattr__ costs half a microsecond per parameter) and held until the call returns.
struct Layer {
    Ref weight, scale, input_scale, layout, granularity, bias, spec;
    bool stream;
};
// Whether calling o.name() would run `fn`: the class's own method, not overridden by the instance.
bool has_method(PyObject* o, PyObject* name, PyObject* fn) {
    PyObject** dp = _PyObject_GetDictPtr(o);
    return _PyType_Lookup(Py_TYPE(o), name) == fn && !(dp && *dp && PyDict_GetItemWithError(*dp, name));
}
PyObject* plain_attr(PyObject* o, PyObject* dict, PyObject* name) {   // instance attribute, else the class's
    PyObject* v = PyDict_GetItemWithError(dict, name);
    return v ? v : _PyType_Lookup(Py_TYPE(o), name);
}
bool layer_of(PyObject* o, Layer* l) {
    PyObject** dp = _PyObject_GetDictPtr(o);
    if (!dp || !*dp) return false;
    PyObject* params = PyDict_GetItemWithError(*dp, s_parameters);
    PyObject* spec = PyDict_GetItemWithError(*dp, s_spec);
    if (!params || !PyDict_Check(params) || !spec) return false;
    l->weight.set(PyDict_GetItemWithError(params, s_weight));
    l->scale.set(PyDict_GetItemWithError(params, s_weight_scale));
    l->input_scale.set(PyDict_GetItemWithError(params, s_input_scale));
    l->bias.set(PyDict_GetItemWithError(params, s_bias));
    if (!l->weight || !l->scale) return false;
    l->layout.set(none_if_null(plain_attr(o, *dp, s_weight_layout)));
    l->spec.set(spec);
    Ref st;
    st.set(plain_attr(o, *dp, s_stream_weights));
    l->stream = st && PyObject_IsTrue(st) == 1;
    l->granularity.p = PyObject_GetAttr(l->spec, s_granularity);
    return l->granularity.p != nullptr;
}

PyObject* layer_call(const Layer& l, PyObject* x, PyObject* bias, int epi, PyObject* residual, PyObject* gate) {
    if (Py_TYPE(x) == (PyTypeObject*)py.view_type) {
        if (l.granularity != py.per_channel || PyTuple_GET_SIZE(x) != 3 || PyTuple_GET_ITEM(x, 2) != py.per_channel) return nullptr;
        return linear_call(PyTuple_GET_ITEM(x, 0), PyTuple_GET_ITEM(x, 1), l.weight, l.scale, bias, epi, l.layout, l.stream, Py_None,
                           residual, gate);
    }
    if (l.granularity == py.per_channel)
        return linear_call(x, nullptr, l.weight, l.scale, bias, epi, l.layout, l.stream, Py_None, residual, gate);
    // (a spec that makes these codes in another way is asked for them, by the Python path)
    if (l.granularity == py.per_tensor && l.input_scale && has_method(l.spec, s_quantize, pl.quantize_activation))
        return linear_static_call(x, l.input_scale, l.weight, l.scale, bias, epi, l.layout, l.stream, residual, gate);
    return nullptr;
}

// layer_apply(layer, x or ActivationView, bias, epilogue, residual, gate)
PyObject* py_layer_apply(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Layer l;
    int epi;
    if (n != 6 || !layer_of(a[0], &l) || !epilogue_of(a[3], &epi)) return declined();
    PyObject* y = layer_call(l, a[1], a[2], epi, a[4], a[5]);
    return y ? y : declined();
    END_HANDLE_TH_ERRORS
}

// Fused epilogues are for layers that say so themselves.
bool own_supports(PyObject* layer) { return has_method(layer, s_supports, pm.linear_supports); }
// Whether the dispatcher's remembered choice (LinearBase._kernel_for, which fills the memory this reads) for
// this layer and input is the HIP kernel with its own apply, which the native calls stand for.  False also where nothing
// is remembered yet.
bool hip_kernel_remembered(PyObject* layer, PyObject* x) {
    PyObject** dp = _PyObject_GetDictPtr(layer);
    if (!dp || !*dp || !pl.mode) return false;
    PyObject* memo = PyDict_GetItemWithError(*dp, s_selected);   // (dispatcher, generation, spec, params_dtype, {key: kernel})
    if (!memo || !PyTuple_CheckExact(memo) || PyTuple_GET_SIZE(memo) != 5) return false;
    PyObject* d = PyDict_GetItemWithError(pl.dispatch_dict, s_dispatcher);
    if (!d || d != PyTuple_GET_ITEM(memo, 0)) return false;
    PyObject** dd = _PyObject_GetDictPtr(d);
    PyObject* gen = dd && *dd ? PyDict_GetItemWithError(*dd, s_generation) : nullptr;
    if (!gen || PyObject_RichCompareBool(gen, PyTuple_GET_ITEM(memo, 1), Py_EQ) != 1) return false;
    PyObject* params_dtype = PyDict_GetItemWithError(*dp, s_params_dtype);
    if (PyDict_GetItemWithError(*dp, s_spec) != PyTuple_GET_ITEM(memo, 2) || params_dtype != PyTuple_GET_ITEM(memo, 3)) return false;
    const bool view = Py_TYPE(x) == (PyTypeObject*)py.view_type;
    const at::Tensor* t = tensor(view && PyTuple_GET_SIZE(x) == 3 ? PyTuple_GET_ITEM(x, 0) : x);
    if (!t || t->dim() < 1 || t->numel() == 0) return false;
    const uint64_t M = (uint64_t)(t->numel() / t->size(t->dim() - 1));
    PyObject* mode = nullptr;
    if (PyContextVar_Get(pl.mode, nullptr, &mode) < 0 || !mode) return false;
    PyObject* bits = PyLong_FromLong(64 - __builtin_clzll(M));
    PyObject* key = PyTuple_Pack(3, bits, view ? params_dtype : (PyObject*)torch::getTHPDtype(t->scalar_type()), mode);
    Py_XDECREF(bits);
    Py_DECREF(mode);
    if (!key) return false;
    PyObject* kernel = PyDict_GetItemWithError(PyTuple_GET_ITEM(memo, 4), key);
    Py_DECREF(key);
    return kernel && Py_TYPE(kernel) == (PyTypeObject*)pl.kernel_type && has_method(kernel, s_apply, pl.kernel_apply);
}
// Whether the layer adds its own bias (None counts as one) or, with skip_bias_add, leaves it to the caller.
enum BiasUse { BIAS_UNKNOWN, BIAS_ADDED, BIAS_LEFT };
BiasUse bias_use(PyObject* layer, const Layer& l) {
    PyObject* skip = PyDict_GetItemWithError(*_PyObject_GetDictPtr(layer), s_skip_bias_add);
    if (!skip || !l.bias) return BIAS_UNKNOWN;
    return skip == Py_False ? BIAS_ADDED : skip == Py_True ? BIAS_LEFT : BIAS_UNKNOWN;
}

// layer_forward(layer, x or ActivationView, epilogue, residual, gate): selection and call in one
PyObject* py_layer_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Layer l;
    int epi;
    if (n != 5 || !hip_kernel_remembered(a[0], a[1]) || !layer_of(a[0], &l) || !epilogue_of(a[2], &epi)) return declined();
    const BiasUse use = bias_use(a[0], l);
    if (use == BIAS_UNKNOWN || (use == BIAS_LEFT && (epi != 0 || a[3] != Py_None)) || (a[3] != Py_None && !own_supports(a[0])))
        return declined();   // fused forms exist for layers that add their own bias
    PyObject* y = layer_call(l, a[1], use == BIAS_ADDED ? l.bias.p : Py_None, epi, a[3], a[4]);
    return y ? y : declined();
    END_HANDLE_TH_ERRORS
}

// ---- MLP ------------------------------------------------------------------------------------------------------------
PyObject* mlp_call(PyObject* x_, PyObject* w1_, PyObject* s1_, PyObject* b1_, PyObject* lay1, bool st1, PyObject* w2_,
                   PyObject* s2_, PyObject* b2_, PyObject* lay2, bool st2, int epi, PyObject* out_, PyObject* res_,
                   PyObject* gate_, PyObject* mod_ = nullptr, PyObject* eps_ = nullptr) {
    const at::Tensor* x = tensor(x_);
    Rows r;
    Where at_;
    Weight w1, w2;
    int f1, f2;
    Residual rg;
    if (!x || epi == 0 || !rows_of(*x, at::kBFloat16, &r) || !where(*x, &at_) || !weight_of(w1_, s1_, b1_, r.K, &w1)) return nullptr;
    if (is_gated(epi) && w1.N % 32 != 0) return nullptr;
    const int64_t I = is_gated(epi) ? w1.N / 2 : w1.N;
    if (!weight_of(w2_, s2_, b2_, I, &w2) || !flags_of(lay1, st1, epi, &f1) || !flags_of(lay2, st2, 0, &f2)) return nullptr;
    Modulation mod = {};
    if (mod_ && !modulation_of(mod_, eps_, r.K, r.M, &mod)) return nullptr;
    if (mod_ ? !residual_gated_by(res_, mod_, *x, r.M, w2.N, &rg) : !residual_of(res_, gate_, *x, r.M, w2.N, 0, &rg)) return nullptr;
    at::Tensor made;
    void* out;
    if (out_ == Py_None) {
        made = fresh(*x, w2.N, at::kBFloat16, at_.dev);
        out = made.mutable_data_ptr();
    } else {
        const at::Tensor* o = tensor(out_);
        if (!shaped(o, *x, w2.N, at::kBFloat16)) return nullptr;
        out = o->mutable_data_ptr();
    }
    Scratch ws;
    if (!workspace(lib.mlp_ws(r.M, r.K, I, w2.N, epi), at_, &ws)) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    if (mod_)
        rc = lib.norm_mlp(r.p, r.ld, mod.p, mod.ld, mod.rows, (float)mod.eps, w1.w, w1.scale, w1.bias, f1, w2.w, w2.scale, w2.bias, f2,
                          rg.residual, w2.N, rg.gate, rg.ld_gate, rg.gate_rows, out, w2.N, r.M, r.K, I, w2.N, epi, ws.p, ws.n, at_.stream);
    else
        rc = lib.mlp(r.p, r.ld, w1.w, w1.scale, w1.bias, f1, w2.w, w2.scale, w2.bias, f2, rg.residual, rg.residual ? w2.N : 0, rg.gate,
                     rg.ld_gate, rg.gate_rows, out, w2.N, r.M, r.K, I, w2.N, epi, ws.p, ws.n, at_.stream);
    Py_END_ALLOW_THREADS
    if (rc != 0) return nullptr;
    if (out_ != Py_None) {
        Py_INCREF(out_);
        return out_;
    }
    return THPVariable_Wrap(std::move(made));
}

// mlp(x, w1, s1, b1, w2, s2, b2, epilogue, out, residual, gate, stream1, stream2, layout1, layout2)
PyObject* py_mlp(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    int epi;
    if (n != 15 || !epilogue_of(a[7], &epi)) return declined();
    PyObject* y = mlp_call(a[0], a[1], a[2], a[3], a[13], PyObject_IsTrue(a[11]) == 1, a[4], a[5], a[6], a[14],
                           PyObject_IsTrue(a[12]) == 1, epi, a[8], a[9], a[10]);
    return y ? y : declined();
    END_HANDLE_TH_ERRORS
}
// both projections per-channel layers that add their own bias
PyObject* mlp_native(PyObject* first, PyObject* second, PyObject* x, int epi, PyObject* residual, PyObject* gate) {
    Layer p, q;
    if (!tensor(x) || !hip_kernel_remembered(first, x) || !hip_kernel_remembered(second, x) || !layer_of(first, &p) || !layer_of(second, &q) ||
        p.granularity != py.per_channel || q.granularity != py.per_channel || bias_use(first, p) != BIAS_ADDED || bias_use(second, q) != BIAS_ADDED ||
        !own_supports(first) || !own_supports(second))
        return nullptr;
    return mlp_call(x, p.weight, p.scale, p.bias, p.layout, p.stream, q.weight, q.scale, q.bias, q.layout, q.stream, epi, Py_None, residual, gate);
}
// mlp_forward(first layer, second layer, x, epilogue, residual, gate)
PyObject* py_mlp_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    int epi;
    PyObject* y = n == 6 && epilogue_of(a[3], &epi) ? mlp_native(a[0], a[1], a[2], epi, a[4], a[5]) : nullptr;
    return y ? y : declined();
    END_HANDLE_TH_ERRORS
}

// ---- loading -------------------------------------------------------------------------------------------------------
// quantize_weight(layer, bf16 [N, K]): codes and scales into the layer's parameters -> True, or None
PyObject* py_quantize_weight(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Layer l;
    if (n != 2 || !layer_of(a[0], &l) || l.granularity != py.per_channel) return declined();
    const at::Tensor *x = tensor(a[1]), *w = tensor(l.weight), *s = tensor(l.scale);
    Where at_;
    if (!x || !w || !s || x->dim() != 2 || w->dim() != 2 || !x->is_cuda() || !w->is_cuda() || x->scalar_type() != at::kBFloat16 || !codes_dtype(*w) ||
        !x->is_contiguous() || !w->is_contiguous() || x->size(0) != w->size(0) || x->size(1) != w->size(1) || x->numel() == 0 ||
        x->size(1) % 8 != 0 || !vector_of(s, at::kFloat, w->size(0)) || x->device() != w->device() || s->device() != w->device() || !where(*x, &at_))
        return declined();
    if (lib.weight_quant(x->const_data_ptr(), x->size(0), x->size(1), x->size(1), w->mutable_data_ptr(), s->mutable_data_ptr<float>(), at_.stream) != 0)
        return declined();
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}
// relay_weight(weight, gated): the matrix re-laid in MFMA operand order, in its own storage -> True, or None
PyObject* py_relay_weight(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor* w = n == 2 ? tensor(a[0]) : nullptr;
    Where at_;
    if (!w || !w->is_cuda() || w->dim() != 2 || !codes_dtype(*w) || !w->is_contiguous() || w->numel() == 0 || !where(*w, &at_)) return declined();
    const int64_t N = w->size(0), K = w->size(1);
    const bool gated = a[1] == Py_True;
    void* p = w->mutable_data_ptr();
    if (!gated && lib.relay_inplace(p, N, K, at_.stream) == 0) Py_RETURN_TRUE;
    at::Tensor t = at::Tensor(at::detail::empty_cuda(w->sizes(), w->scalar_type(), at_.dev, std::nullopt));
    if (gated) {
        const int rc = lib.relay_gated(p, N, K, t.mutable_data_ptr(), at_.stream);
        if (rc == 0) Py_RETURN_TRUE;
        TORCH_CHECK(rc == -2, "relay_weight: a launch failed");   // (half of the matrix is re-laid)
    }
    // (a plain copy first and the re-lay back: the allocator's stream order covers the temporary)
    if (hipMemcpyAsync(t.mutable_data_ptr(), p, (size_t)(N * K), hipMemcpyDeviceToDevice, at_.stream) != hipSuccess) return declined();
    if (lib.relay(t.const_data_ptr(), N, K, gated, p, at_.stream) != 0) return declined();
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// ---- a decoder layer's three calls: adaptive norm + linear, linear + gated residual, adaptive norm + MLP + gated residual
// norm_linear(layer, x, modulation, eps): layer(norm(x)), x in rows of the layer's input width
PyObject* py_norm_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Layer l;
    if (n != 4 || !hip_kernel_remembered(a[0], a[1]) || !layer_of(a[0], &l) || l.granularity != py.per_channel || bias_use(a[0], l) != BIAS_ADDED)
        return declined();
    PyObject* y = linear_call(a[1], nullptr, l.weight, l.scale, l.bias, 0, l.layout, l.stream, Py_None, Py_None, Py_None, false, a[2], a[3]);
    return y ? y : declined();
    END_HANDLE_TH_ERRORS
}
// linear_residual(layer, x, residual, modulation): residual + layer(x) * gate part of the modulation
PyObject* py_linear_residual(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Layer l;
    if (n != 4 || !hip_kernel_remembered(a[0], a[1]) || !layer_of(a[0], &l) || l.granularity != py.per_channel || bias_use(a[0], l) != BIAS_ADDED)
        return declined();
    PyObject* y = linear_call(a[1], nullptr, l.weight, l.scale, l.bias, 0, l.layout, l.stream, Py_None, a[2], a[3], true);
    return y ? y : declined();
    END_HANDLE_TH_ERRORS
}
// norm_mlp(first layer, second layer, x, modulation, eps, epilogue): x + mlp(norm(x)) * gate part of the modulation
PyObject* py_norm_mlp(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Layer p, q;
    int epi;
    if (n != 6 || !tensor(a[2]) || !hip_kernel_remembered(a[0], a[2]) || !hip_kernel_remembered(a[1], a[2]) || !layer_of(a[0], &p) ||
        !layer_of(a[1], &q) || !epilogue_of(a[5], &epi) || p.granularity != py.per_channel || q.granularity != py.per_channel ||
        bias_use(a[0], p) != BIAS_ADDED || bias_use(a[1], q) != BIAS_ADDED)
        return declined();
    PyObject* y = mlp_call(a[2], p.weight, p.scale, p.bias, p.layout, p.stream, q.weight, q.scale, q.bias, q.layout, q.stream, epi, Py_None,
                           a[2], nullptr, a[3], a[4]);
    return y ? y : declined();
    END_HANDLE_TH_ERRORS
}

// ---- modules: __call__ of the linear layers and of the MLP ---------------------------------------------------------
// nn.Module.__call__ and the two Python frames behind it take 0.9 us.  These go straight to the native call when nothing
// stands in between - no hooks, no compiled or replaced forward - and to nn.Module.__call__ otherwise.
bool plain_call(PyObject* self, PyObject* dict, PyObject* forward) {
    if (!pm.self || PyDict_GetItemWithError(pm.ops_dict, s_host) != pm.self) return false;
    if (_PyType_Lookup((PyTypeObject*)pm.module_type, s_call) != pm.module_call) return false;   // replaced, as torch.fx does while it traces
    if (_PyType_Lookup(Py_TYPE(self), s_forward) != forward || PyDict_GetItemWithError(dict, s_forward) || PyDict_GetItemWithError(dict, s_compiled))
        return false;
    for (PyObject* name : s_hooks) {
        PyObject* h = PyDict_GetItemWithError(dict, name);
        if (!h || !PyDict_Check(h) || PyDict_GET_SIZE(h) != 0) return false;
    }
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(pm.global_hooks); ++i)
        if (PyDict_GET_SIZE(PyTuple_GET_ITEM(pm.global_hooks, i)) != 0) return false;
    return true;
}
PyObject* module_call(PyObject* args, PyObject* kwargs) {   // nn.Module.__call__ as it is now
    PyErr_Clear();
    Ref call;
    call.p = PyObject_GetAttr(pm.module_type, s_call);
    return call ? PyObject_Call(call, args, kwargs) : nullptr;
}
// decoder_layer_plain(qkv_proj, o_proj, gate_up_proj, down_proj, first norm, second norm): whether the three calls above
// do what these parts' own methods would - qkv_proj called as a module (hooks, a replaced forward, a wrapper around
// it), the others through the methods that a decoder layer uses of them
PyObject* py_decoder_layer_plain(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 6) return PyErr_Format(PyExc_TypeError, "six parts");
    PyObject** dp = _PyObject_GetDictPtr(a[0]);
    const bool plain = pm.self && dp && *dp && _PyType_Lookup(Py_TYPE(a[0]), s_call) == pm.linear_call && plain_call(a[0], *dp, pm.linear_forward) &&
                       has_method(a[1], s_forward_addcmul, pm.linear_forward_addcmul) && has_method(a[2], s_forward_fused, pm.linear_forward_fused) &&
                       has_method(a[3], s_forward_addcmul, pm.linear_forward_addcmul) && has_method(a[4], s_forward_fp8, pm.norm_forward_fp8) &&
                       has_method(a[5], s_forward_fp8, pm.norm_forward_fp8) && own_supports(a[1]) && own_supports(a[3]);
    if (PyErr_Occurred()) return nullptr;
    return PyBool_FromLong(plain);
}
// linear(x) -> (output, bias left to the caller or None)
PyObject* py_linear_call(PyObject*, PyObject* args, PyObject* kwargs) {
    HANDLE_TH_ERRORS
    if (PyTuple_GET_SIZE(args) == 2 && (!kwargs || PyDict_GET_SIZE(kwargs) == 0)) {
        PyObject *self = PyTuple_GET_ITEM(args, 0), *x = PyTuple_GET_ITEM(args, 1);
        PyObject** dp = _PyObject_GetDictPtr(self);
        Layer l;
        if (dp && *dp && plain_call(self, *dp, pm.linear_forward) && hip_kernel_remembered(self, x) && layer_of(self, &l)) {
            const BiasUse use = bias_use(self, l);
            PyObject* y = use == BIAS_UNKNOWN ? nullptr : layer_call(l, x, use == BIAS_ADDED ? l.bias.p : Py_None, 0, Py_None, Py_None);
            if (y) {
                PyObject* r = PyTuple_Pack(2, y, use == BIAS_LEFT ? l.bias.p : Py_None);
                Py_DECREF(y);
                return r;
            }
        }
    }
    return module_call(args, kwargs);
    END_HANDLE_TH_ERRORS
}
// mlp(x, residual=, gate=)
PyObject* py_mlp_call(PyObject*, PyObject* args, PyObject* kwargs) {
    HANDLE_TH_ERRORS
    if (PyTuple_GET_SIZE(args) == 2) {
        PyObject *self = PyTuple_GET_ITEM(args, 0), *x = PyTuple_GET_ITEM(args, 1), *residual = Py_None, *gate = Py_None;
        Py_ssize_t known = 0;
        if (kwargs) {
            if (PyObject* r = PyDict_GetItemWithError(kwargs, s_residual)) { residual = r; ++known; }
            if (PyObject* g = PyDict_GetItemWithError(kwargs, s_gate)) { gate = g; ++known; }
        }
        PyObject** dp = _PyObject_GetDictPtr(self);
        if ((!kwargs || known == PyDict_GET_SIZE(kwargs)) && dp && *dp && plain_call(self, *dp, pm.mlp_forward) &&
            PyDict_GetItemWithError(*dp, s_fuse_activation) == Py_True) {
            PyObject *mods = PyDict_GetItemWithError(*dp, s_modules), *epilogue = PyDict_GetItemWithError(*dp, s_epilogue);
            const bool gated = PyDict_GetItemWithError(*dp, s_gated) == Py_True;
            Ref first, second;
            first.set(mods ? PyDict_GetItemWithError(mods, gated ? s_gate_up : s_fc1) : nullptr);
            second.set(mods ? PyDict_GetItemWithError(mods, gated ? s_down : s_fc2) : nullptr);
            int epi;
            if (first && second && epilogue && epilogue_of(epilogue, &epi)) {
                PyObject* y = mlp_native(first, second, x, epi, residual, gate);
                if (y) return y;
            }
        }
    }
    return module_call(args, kwargs);
    END_HANDLE_TH_ERRORS
}

// ---- quantizers and norms ------------------------------------------------------------------------------------------
// quant_rowwise(x) -> (codes, scale)
PyObject* py_quant_rowwise(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor* x = n == 1 ? tensor(a[0]) : nullptr;
    Rows r;
    Where at_;
    if (!x || !rows_of(*x, at::kBFloat16, &r) || r.K % 8 != 0 || !where(*x, &at_)) return declined();
    at::Tensor q = fresh(*x, r.K, at::kFloat8_e4m3fn, at_.dev), s = fresh(*x, 1, at::kFloat, at_.dev);
    if (lib.quant_rowwise(r.p, r.M, r.K, r.ld, q.mutable_data_ptr(), s.mutable_data_ptr<float>(), at_.stream) != 0) return declined();
    return Py_BuildValue("NN", THPVariable_Wrap(std::move(q)), THPVariable_Wrap(std::move(s)));
    END_HANDLE_TH_ERRORS
}

struct NormOut {
    at::Tensor out, xq, xs;
    void* out_p() { return out.defined() ? out.mutable_data_ptr() : nullptr; }
    void* xq_p() { return xq.defined() ? xq.mutable_data_ptr() : nullptr; }
    float* xs_p() { return xs.defined() ? xs.mutable_data_ptr<float>() : nullptr; }
};
void make_norm_outputs(const at::Tensor& x, int64_t D, bool quantize, bool want_out, const Where& w, NormOut* o) {
    if (want_out) o->out = fresh(x, D, at::kBFloat16, w.dev);
    if (quantize) {
        o->xq = fresh(x, D, at::kFloat8_e4m3fn, w.dev);
        o->xs = fresh(x, 1, at::kFloat, w.dev);
    }
}
PyObject* wrap_or_none(at::Tensor& t) {
    if (t.defined()) return THPVariable_Wrap(std::move(t));
    Py_RETURN_NONE;
}

// rmsnorm(x, weight, eps, gemma, quantize, want_out) -> (out, codes, scale)
PyObject* py_rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor *x = n == 6 ? tensor(a[0]) : nullptr, *w = n == 6 ? tensor(a[1]) : nullptr;
    Rows r;
    Where at_;
    if (!x || !w || !rows_of(*x, at::kBFloat16, &r) || r.K % 8 != 0 || w->dim() != 1 || !vector_of(w, at::kBFloat16, r.K) || !where(*x, &at_))
        return declined();
    const double eps = PyFloat_AsDouble(a[2]);
    if (eps == -1.0 && PyErr_Occurred()) return declined();
    NormOut o;
    make_norm_outputs(*x, r.K, a[4] == Py_True, a[5] == Py_True, at_, &o);
    if (lib.rmsnorm(r.p, r.ld, w->const_data_ptr(), a[3] == Py_True, r.M, r.K, (float)eps, o.out_p(), r.K, o.xq_p(), o.xs_p(), at_.stream) != 0)
        return declined();
    return Py_BuildValue("NNN", wrap_or_none(o.out), wrap_or_none(o.xq), wrap_or_none(o.xs));
    END_HANDLE_TH_ERRORS
}

PyObject* view_of(at::Tensor& xq, at::Tensor& xs) {
    PyObject *q = THPVariable_Wrap(std::move(xq)), *s = THPVariable_Wrap(std::move(xs));
    PyObject* v = q && s ? PyObject_CallFunctionObjArgs(py.view_type, q, s, py.per_channel, nullptr) : nullptr;
    Py_XDECREF(q);
    Py_XDECREF(s);
    return v;
}

// adarmsnorm(x, modulation, eps, quantize, want_out) -> (out, codes, scale, gate)
// adarmsnorm(x, modulation, eps, True, False, hidden size) -> (ActivationView, gate), the rows of x and modulation
// checked against the hidden size and (B, 3D) modulation rows serving the (S, D) rows of each item of the batch
PyObject* py_adarmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor *x = n >= 5 ? tensor(a[0]) : nullptr, *m = n >= 5 ? tensor(a[1]) : nullptr;
    if (n == 6 && (!x || !m || x->dim() != 2 || m->dim() != 2 || x->size(1) != PyLong_AsLong(a[5]))) return declined();
    Rows r, q;
    Where at_;
    if (!x || !m || !rows_of(*x, at::kBFloat16, &r) || !rows_of(*m, at::kBFloat16, &q) || r.K % 8 != 0 || q.K != 3 * r.K ||
        r.M % q.M != 0 || !where(*x, &at_))
        return declined();
    const double eps = PyFloat_AsDouble(a[2]);
    if (eps == -1.0 && PyErr_Occurred()) return declined();
    NormOut o;
    make_norm_outputs(*x, r.K, a[3] == Py_True, a[4] == Py_True, at_, &o);
    at::Tensor gate = fresh(*m, r.K, at::kBFloat16, at_.dev);
    if (lib.adarmsnorm(r.p, r.ld, q.p, q.M > 1 ? q.ld : q.K, q.M, r.M, r.K, (float)eps, o.out_p(), r.K, gate.mutable_data_ptr(), r.K,
                       o.xq_p(), o.xs_p(), at_.stream) != 0)
        return declined();
    if (n == 6) return Py_BuildValue("NN", view_of(o.xq, o.xs), THPVariable_Wrap(std::move(gate)));
    return Py_BuildValue("NNNN", wrap_or_none(o.out), wrap_or_none(o.xq), wrap_or_none(o.xs), THPVariable_Wrap(std::move(gate)));
    END_HANDLE_TH_ERRORS
}

// ---- module --------------------------------------------------------------------------------------------------------
// bind(library path, workspaces, owner variable, reserve, epilogues, layouts, ActivationView, PER_CHANNEL, PER_TENSOR)
PyObject* py_bind(PyObject*, PyObject* args) {
    const char* path;
    Py p = {};
    if (!PyArg_ParseTuple(args, "sOOOOOOOO", &path, &p.workspaces, &p.owner, &p.reserve, &p.epilogues, &p.layouts, &p.view_type,
                          &p.per_channel, &p.per_tensor))
        return nullptr;
    void* h = dlopen(path, RTLD_NOW | RTLD_LOCAL);   // the library that is loaded already: one more reference to it
    if (!h) return PyErr_Format(PyExc_RuntimeError, "%s", dlerror());
    Lib l = {};
    bool ok = true;
    auto get = [&](auto& fn, const char* name) {
        fn = reinterpret_cast<std::decay_t<decltype(fn)>>(dlsym(h, name));
        ok = ok && fn != nullptr;
    };
    get(l.linear, "phyai_fp8_linear");
    get(l.linear_addcmul, "phyai_fp8_linear_addcmul");
    get(l.gemm, "phyai_fp8_gemm");
    get(l.gemm_addcmul, "phyai_fp8_gemm_addcmul");
    get(l.mlp, "phyai_fp8_mlp");
    get(l.norm_linear, "phyai_fp8_adarmsnorm_linear");
    get(l.norm_mlp, "phyai_fp8_adarmsnorm_mlp");
    get(l.linear_ws, "phyai_fp8_linear_workspace_bytes");
    get(l.mlp_ws, "phyai_fp8_mlp_workspace_bytes");
    get(l.quant_rowwise, "phyai_fp8_quant_rowwise");
    get(l.weight_quant, "phyai_fp8_weight_quant_rowwise");
    get(l.relay, "phyai_fp8_weight_to_operand_order");
    get(l.relay_inplace, "phyai_fp8_weight_to_operand_order_inplace");
    get(l.relay_gated, "phyai_host_relay_gated");
    get(l.per_tensor, "phyai_fp8_linear_per_tensor");
    get(l.rmsnorm, "phyai_fp8_rmsnorm_quant");
    get(l.adarmsnorm, "phyai_fp8_adarmsnorm_quant");
    if (!ok) return PyErr_Format(PyExc_RuntimeError, "%s lacks an entry point this extension binds", path);
    for (PyObject* o : {p.workspaces, p.owner, p.reserve, p.epilogues, p.layouts, p.view_type, p.per_channel, p.per_tensor}) Py_INCREF(o);
    lib = l;
    py = p;
    Py_RETURN_NONE;
}

// bind_layers(phyai_amd.linear.dispatch's dictionary, mode variable, HipFp8Kernel, its apply, Fp8Spec.quantize_activation)
PyObject* py_bind_layers(PyObject*, PyObject* args) {
    PyLayers p = {};
    if (!PyArg_ParseTuple(args, "O!OOOO", &PyDict_Type, &p.dispatch_dict, &p.mode, &p.kernel_type, &p.kernel_apply, &p.quantize_activation))
        return nullptr;
    for (PyObject* o : {p.dispatch_dict, p.mode, p.kernel_type, p.kernel_apply, p.quantize_activation}) Py_INCREF(o);
    pl = p;
    Py_RETURN_NONE;
}

PyMethodDef linear_call_def = {"__call__", (PyCFunction)(void (*)(void))py_linear_call, METH_VARARGS | METH_KEYWORDS, nullptr};
PyMethodDef mlp_call_def = {"__call__", (PyCFunction)(void (*)(void))py_mlp_call, METH_VARARGS | METH_KEYWORDS, nullptr};
// bind_modules(phyai_amd.ops's dictionary, this module, nn.Module, its own __call__, tuple of global hook tables,
//              LinearBase.forward, DenseMLP.forward, LinearBase.forward_fused, .forward_addcmul,
//              .supports_fused_epilogue, AdaRMSNorm.forward_fp8)
//   -> (LinearBase.__call__, DenseMLP.__call__)
PyObject* py_bind_modules(PyObject*, PyObject* args) {
    PyModules m = {};
    if (!PyArg_ParseTuple(args, "O!OO!OO!OOOOOO", &PyDict_Type, &m.ops_dict, &m.self, &PyType_Type, &m.module_type, &m.module_call, &PyTuple_Type,
                          &m.global_hooks, &m.linear_forward, &m.mlp_forward, &m.linear_forward_fused, &m.linear_forward_addcmul,
                          &m.linear_supports, &m.norm_forward_fp8))
        return nullptr;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(m.global_hooks); ++i)
        if (!PyDict_Check(PyTuple_GET_ITEM(m.global_hooks, i))) return PyErr_Format(PyExc_TypeError, "hook tables are dictionaries");
    for (PyObject* o : {m.ops_dict, m.self, m.module_type, m.module_call, m.global_hooks, m.linear_forward, m.mlp_forward, m.linear_forward_fused,
                        m.linear_forward_addcmul, m.linear_supports, m.norm_forward_fp8})
        Py_INCREF(o);
    PyObject *a = PyCFunction_New(&linear_call_def, nullptr), *b = PyCFunction_New(&mlp_call_def, nullptr);
    PyObject *ma = a ? PyInstanceMethod_New(a) : nullptr, *mb = b ? PyInstanceMethod_New(b) : nullptr;
    Py_XDECREF(a);
    Py_XDECREF(b);
    Py_XINCREF(ma);
    m.linear_call = ma;
    pm = m;
    return ma && mb ? Py_BuildValue("NN", ma, mb) : nullptr;
}

#define PHYAI_FAST(name, fn) {name, (PyCFunction)(void (*)(void))fn, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", py_bind, METH_VARARGS, nullptr},
    {"bind_layers", py_bind_layers, METH_VARARGS, nullptr},
    {"bind_modules", py_bind_modules, METH_VARARGS, nullptr},
    PHYAI_FAST("linear", py_linear),
    PHYAI_FAST("gemm", py_gemm),
    PHYAI_FAST("mlp", py_mlp),
    PHYAI_FAST("layer_apply", py_layer_apply),
    PHYAI_FAST("layer_forward", py_layer_forward),
    PHYAI_FAST("mlp_forward", py_mlp_forward),
    PHYAI_FAST("quantize_weight", py_quantize_weight),
    PHYAI_FAST("relay_weight", py_relay_weight),
    PHYAI_FAST("norm_linear", py_norm_linear),
    PHYAI_FAST("linear_residual", py_linear_residual),
    PHYAI_FAST("norm_mlp", py_norm_mlp),
    PHYAI_FAST("decoder_layer_plain", py_decoder_layer_plain),
    PHYAI_FAST("quant_rowwise", py_quant_rowwise),
    PHYAI_FAST("rmsnorm", py_rmsnorm),
    PHYAI_FAST("adarmsnorm", py_adarmsnorm),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_phyai_host", "Eager call path of phyai_amd.ops and of the fp8 layers.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__phyai_host() {
    const struct { PyObject** at; const char* text; } names[] = {
        {&s_parameters, "_parameters"}, {&s_weight, "weight"}, {&s_weight_scale, "weight_scale"}, {&s_input_scale, "input_scale"},
        {&s_stream_weights, "stream_weights"}, {&s_weight_layout, "weight_layout"}, {&s_spec, "spec"},
        {&s_granularity, "granularity"}, {&s_apply, "apply"}, {&s_quantize, "quantize_activation"},
        {&s_dispatcher, "_dispatcher"}, {&s_generation, "generation"}, {&s_selected, "_selected"},
        {&s_params_dtype, "params_dtype"}, {&s_skip_bias_add, "skip_bias_add"}, {&s_bias, "bias"}, {&s_host, "_host"},
        {&s_call, "__call__"}, {&s_forward, "forward"}, {&s_forward_fused, "forward_fused"}, {&s_forward_addcmul, "forward_addcmul"},
        {&s_forward_fp8, "forward_fp8"}, {&s_supports, "supports_fused_epilogue"},
        {&s_fuse_activation, "fuse_activation"}, {&s_gated, "gated"}, {&s_epilogue, "_epilogue"}, {&s_modules, "_modules"},
        {&s_gate_up, "gate_up_proj"}, {&s_down, "down_proj"}, {&s_fc1, "fc1"}, {&s_fc2, "fc2"}, {&s_residual, "residual"}, {&s_gate, "gate"},
        {&s_compiled, "_compiled_call_impl"}, {&s_hooks[0], "_forward_hooks"}, {&s_hooks[1], "_forward_pre_hooks"},
        {&s_hooks[2], "_backward_hooks"}, {&s_hooks[3], "_backward_pre_hooks"}};
    for (const auto& e : names)
        if (!(*e.at = PyUnicode_InternFromString(e.text))) return nullptr;
    return PyModule_Create(&module);
}
