// The operators' host path as native code (a CPython extension over libtorch): argument checks, output and workspace allocation and
// the call into libgdn_hip.so for the calls that need no conversion of any kind - every tensor contiguous, aligned, on the current
// device and of a type and shape the kernels take as it is.  Every function returns None for anything else (wrong arguments
// included) and changes nothing then: the Python path behind it converts, pads or raises.  What fails inside (no memory left, a library
// call refused) leaves as a Python exception of the type torch itself would raise: every entry is a body in torch's own translation.
//
// A call through Python and ctypes took 25 us of host time (decode step) to 60 us (prefill), more than the kernels of a small call.
#include <Python.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "../../../include/gdn_hip.h"

namespace {

// ---- entry points of libgdn_hip.so, handed over by the Python binding that has loaded it ----
decltype(&gdn_fused_recurrent_fwd) p_fused_recurrent_fwd;
decltype(&gdn_fused_recurrent_kda_fwd) p_fused_recurrent_kda_fwd;
decltype(&gdn_chunk_fwd) p_chunk_fwd;
decltype(&gdn_chunk_workspace_bytes) p_chunk_workspace_bytes;
decltype(&gdn_step_linear) p_step_linear;
decltype(&gdn_norm_gated_fwd) p_norm_gated_fwd;
decltype(&gdn_norm_gated_bwd) p_norm_gated_bwd;
decltype(&gdn_chunk_bwd_heads) p_chunk_bwd_heads;
decltype(&gdn_chunk_bwd_heads_workspace_bytes) p_chunk_bwd_heads_workspace_bytes;
decltype(&gdn_causal_conv1d_fwd) p_conv_fwd;
decltype(&gdn_causal_conv1d_bwd_runs) p_conv_bwd_runs;
decltype(&gdn_gate_bwd) p_gate_bwd;
decltype(&gdn_sum_rows) p_sum_rows;
decltype(&gdn_last_error) p_last_error;

PyObject* bind(PyObject*, PyObject* table) {
    HANDLE_TH_ERRORS
    auto take = [&](const char* name, auto& fn) {
        PyObject* at = PyDict_GetItemString(table, name);
        if (!at) { PyErr_Format(PyExc_KeyError, "gdn_host.bind: no address of %s", name); return false; }
        fn = (std::remove_reference_t<decltype(fn)>)PyLong_AsVoidPtr(at);
        return !PyErr_Occurred();
    };
    if (!take("gdn_fused_recurrent_fwd", p_fused_recurrent_fwd) || !take("gdn_fused_recurrent_kda_fwd", p_fused_recurrent_kda_fwd) ||
        !take("gdn_chunk_fwd", p_chunk_fwd) || !take("gdn_chunk_workspace_bytes", p_chunk_workspace_bytes) ||
        !take("gdn_step_linear", p_step_linear) || !take("gdn_norm_gated_fwd", p_norm_gated_fwd) || !take("gdn_norm_gated_bwd", p_norm_gated_bwd) ||
        !take("gdn_chunk_bwd_heads", p_chunk_bwd_heads) || !take("gdn_chunk_bwd_heads_workspace_bytes", p_chunk_bwd_heads_workspace_bytes) ||
        !take("gdn_causal_conv1d_fwd", p_conv_fwd) || !take("gdn_causal_conv1d_bwd_runs", p_conv_bwd_runs) || !take("gdn_gate_bwd", p_gate_bwd) ||
        !take("gdn_sum_rows", p_sum_rows) || !take("gdn_last_error", p_last_error))
        return nullptr;
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// The interpreter runs other threads while this lives (exceptions on their way out take it back).
struct NoGil {
    PyThreadState* state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
    NoGil() = default;
    NoGil(const NoGil&) = delete;
    NoGil& operator=(const NoGil&) = delete;
};

// ---- arguments ----
// Strided memory behind it: not the tensors of tracing, vmap and the other transforms, of subclasses with a dispatch of their own, and
// none that is sparse, nested or to be negated when it is read (the Python path says what becomes of those).  One load
// and one test of a tensor's keys: every call asks this of every tensor.
const uint64_t KEYS_WITHOUT_MEMORY =
    c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::Negative, c10::DispatchKey::Conjugate, c10::DispatchKey::ZeroTensor,
                         c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                         c10::DispatchKey::Sparse, c10::DispatchKey::SparseCsr, c10::DispatchKey::NestedTensor, c10::DispatchKey::MkldnnCPU})
        .raw_repr() & ~c10::full_backend_mask;
inline bool has_memory(const at::Tensor& t) { return (t.unsafeGetTensorImpl()->key_set().raw_repr() & KEYS_WITHOUT_MEMORY) == 0; }

// A tensor argument: absent (None), present, or something else.
struct Arg {
    const at::Tensor* t = nullptr;
    bool bad = false;
    explicit Arg(PyObject* o) {
        if (o == Py_None) return;
        if (THPVariable_Check(o) && has_memory(THPVariable_Unpack(o))) t = &THPVariable_Unpack(o);
        else bad = true;
    }
    explicit operator bool() const { return t != nullptr; }
    const at::Tensor* operator->() const { return t; }
    void* ptr() const { return t ? t->data_ptr() : nullptr; }
};

int code_of(at::ScalarType s) {
    switch (s) {
        case at::kBFloat16: return GDN_DTYPE_BF16;
        case at::kHalf: return GDN_DTYPE_F16;
        case at::kFloat: return GDN_DTYPE_F32;
        default: return -1;
    }
}

bool plain(const Arg& a, c10::Device dev) { return !a.bad && (!a || (a->device() == dev && a->is_contiguous())); }
bool aligned16(const void* p) { return (uintptr_t)p % 16 == 0; }
bool truth(PyObject* o) {                                // (may run the caller's code: with the interpreter held, and it may raise)
    const int is = PyObject_IsTrue(o);
    if (is < 0) throw python_error();
    return is;
}

// g and beta share a code, or carry one each; -1: a type the kernels do not take
int gb_code_of(const Arg& g, const Arg& beta) {
    const int cg = g ? code_of(g->scalar_type()) : -2, cb = beta ? code_of(beta->scalar_type()) : -2;
    if (cg == -1 || cb == -1) return -1;
    if (cg == -2) return cb == -2 ? GDN_DTYPE_F32 : cb;
    return cb == -2 || cb == cg ? cg : GDN_GB_DTYPES(cg, cb);
}

// q, k [B,T,H,K], v [B,T,HV,V] of one type, on the current GPU
struct Dims { int64_t B, T, H, HV, K, V; c10::Device dev{c10::kCPU}; int code; };
bool operands(const Arg& q, const Arg& k, const Arg& v, Dims& d) {
    if (!q || !k || !v || !q->is_cuda() || q->dim() != 4 || v->dim() != 4 || k->sizes() != q->sizes()) return false;
    d.dev = q->device();
    if (!plain(q, d.dev) || !plain(k, d.dev) || !plain(v, d.dev)) return false;
    if (q->scalar_type() != k->scalar_type() || q->scalar_type() != v->scalar_type()) return false;
    d.code = code_of(q->scalar_type());
    d.B = q->size(0); d.T = q->size(1); d.H = q->size(2); d.K = q->size(3); d.HV = v->size(2); d.V = v->size(3);
    return d.code >= 0 && d.B > 0 && d.T > 0 && d.H > 0 && d.K > 0 && d.HV > 0 && d.V > 0 && v->size(0) == d.B && v->size(1) == d.T &&
           d.HV % d.H == 0 && d.dev.index() == c10::hip::current_device();
}
bool per_head(const Arg& x, const Dims& d) {            // [B,T,HV] (or absent)
    return !x || (x->numel() == d.B * d.T * d.HV && x->dim() == 3 && x->size(0) == d.B && x->size(1) == d.T);
}
bool floats(const Arg& x, int64_t n) { return !x || (x->scalar_type() == at::kFloat && x->numel() == n); }
bool indices(const Arg& x, int64_t n) {
    return !x || (x->dim() == 1 && (n < 0 || x->numel() == n) && (x->scalar_type() == at::kLong || x->scalar_type() == at::kInt));
}
bool scale_of(PyObject* o, int64_t K, float& scale) {
    if (o == Py_None) { scale = (float)std::pow((double)K, -0.5); return true; }
    if (!PyFloat_Check(o) && !PyLong_Check(o)) return false;
    scale = (float)PyFloat_AsDouble(o);
    return !PyErr_Occurred();
}
at::Tensor empty_on(c10::Device dev, at::ScalarType s, at::IntArrayRef sizes) { return at::empty(sizes, at::TensorOptions().dtype(s).device(dev)); }
void* stream_of(c10::Device dev) { return (void*)c10::hip::getCurrentHIPStream(dev.index()).stream(); }

PyObject* pair(const at::Tensor& a, const at::Tensor& b) {
    PyObject* x = THPVariable_Wrap(a);
    PyObject* y = b.defined() ? THPVariable_Wrap(b) : (Py_INCREF(Py_None), Py_None);
    PyObject* r = x && y ? PyTuple_Pack(2, x, y) : nullptr;
    Py_XDECREF(x); Py_XDECREF(y);
    return r;
}

// a refusal or a failed launch of the library as the exception that _lib.check raises for it
void check_rc(int rc, const char* what) {
    if (rc == GDN_OK) return;
    const char* why = p_last_error ? p_last_error() : "";
    TORCH_CHECK_VALUE(rc != GDN_ERR_INVALID, what, ": ", why);
    TORCH_CHECK_NOT_IMPLEMENTED(rc != GDN_ERR_UNSUPPORTED, what, ": ", why);
    TORCH_CHECK(false, what, ": libgdn_hip status ", rc, ": ", why);
}

// ---- token recurrence ----
// (q, k, v, g, gk, beta, A_log, dt_bias, scale, initial_state, output_final_state, qk_l2norm, beta_sigmoid, neg_eigval, state_v_first,
//  cu_seqlens, inplace_final_state, state_slots, kda_gate_mode, lower_bound); gk: the KDA operator's gate (kda_gate_mode 0 .. 2) or
// the general operator's log decays per key feature (kda_gate_mode None)
PyObject* fused_recurrent(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 20) { PyErr_SetString(PyExc_TypeError, "gdn_host.fused_recurrent takes 20 arguments"); return nullptr; }
    const Arg q(a[0]), k(a[1]), v(a[2]), g(a[3]), gk(a[4]), beta(a[5]), A_log(a[6]), dt_bias(a[7]), h0(a[9]), cu(a[15]), slots(a[17]);
    const bool out_final = truth(a[10]), bsig = truth(a[12]), neg = truth(a[13]), vfirst = truth(a[14]), inplace = truth(a[16]);
    const bool kda = a[18] != Py_None;
    Dims d;
    float scale;
    if (!operands(q, k, v, d) || !scale_of(a[8], d.K, scale)) Py_RETURN_NONE;
    for (const Arg* x : {&g, &gk, &beta, &A_log, &dt_bias, &h0, &cu, &slots})
        if (!plain(*x, d.dev)) Py_RETURN_NONE;
    if (d.K % 4 || d.V % 4 || d.K > 256 || !per_head(g, d) || !indices(cu, -1) || (neg && !bsig)) Py_RETURN_NONE;
    uint32_t flags = (truth(a[11]) ? GDN_FLAG_QK_L2NORM : 0) | (bsig ? GDN_FLAG_BETA_SIGMOID : 0) | (neg ? GDN_FLAG_NEG_EIGVAL : 0) |
                     (vfirst ? GDN_FLAG_STATE_V_FIRST : 0);
    if (beta && beta->dim() == 4 && beta->sizes() == v->sizes() && d.V > 1) flags |= GDN_FLAG_BETA_VECTOR;
    else if (!per_head(beta, d)) Py_RETURN_NONE;
    if (gk && (gk->scalar_type() != at::kFloat || gk->numel() != d.B * d.T * d.HV * d.K || gk->dim() != 4 || gk->size(2) != d.HV ||
               gk->size(1) != d.T || gk->size(3) != d.K || !aligned16(gk.ptr())))
        Py_RETURN_NONE;
    if (!floats(A_log, d.HV) || !floats(dt_bias, kda ? d.HV * d.K : d.HV) || (dt_bias && !A_log && !kda) || (A_log && !g && !kda)) Py_RETURN_NONE;
    const int gb = gb_code_of(g, beta);
    if (gb < 0) Py_RETURN_NONE;
    const int64_t N = cu ? cu->numel() - 1 : d.B;
    if (N < 1 || (cu && d.B != 1)) Py_RETURN_NONE;
    if (cu && cu->scalar_type() == at::kInt) flags |= GDN_FLAG_CU_INT32;
    if (slots) {
        if (!inplace || !h0 || !indices(slots, N)) Py_RETURN_NONE;
        if (slots->scalar_type() == at::kInt) flags |= GDN_FLAG_SLOT_INT32;
    }
    if (inplace && !h0) Py_RETURN_NONE;
    const int64_t rows = vfirst ? d.V : d.K, cols = vfirst ? d.K : d.V;
    if (h0) {
        if (h0->dim() != 4 || (!slots && h0->size(0) != N) || h0->size(1) != d.HV || h0->size(2) != rows || h0->size(3) != cols || !aligned16(h0.ptr()))
            Py_RETURN_NONE;
        if (h0->scalar_type() == at::kBFloat16) {
            if (!inplace || d.K != 128 || d.V != 128 || vfirst || gk || kda || (flags & GDN_FLAG_BETA_VECTOR)) Py_RETURN_NONE;
            flags |= GDN_FLAG_STATE_BF16;
        } else if (h0->scalar_type() != at::kFloat) Py_RETURN_NONE;
    }
    float lower = 0.f;
    int mode = 0;
    if (kda) {
        if (g || !gk) Py_RETURN_NONE;
        mode = (int)PyLong_AsLong(a[18]);
        lower = (float)PyFloat_AsDouble(a[19]);
        if (PyErr_Occurred()) return nullptr;
    }
    const at::Tensor o = empty_on(d.dev, v->scalar_type(), v->sizes());
    at::Tensor ht;
    if (inplace) ht = *h0.t;
    else if (out_final) ht = empty_on(d.dev, at::kFloat, {N, d.HV, rows, cols});
    void* stream = stream_of(d.dev);
    float* pht = ht.defined() ? (float*)ht.data_ptr() : nullptr;
    int rc;
    {
        const NoGil free;
        if (kda)
            rc = p_fused_recurrent_kda_fwd(q.ptr(), k.ptr(), v.ptr(), (const float*)gk.ptr(), beta.ptr(), (const float*)A_log.ptr(), (const float*)dt_bias.ptr(),
                                           lower, mode, (const float*)h0.ptr(), pht, o.data_ptr(), cu.ptr(), slots.ptr(), nullptr, 1,
                                           d.B, d.T, d.H, d.HV, d.K, d.V, N, scale, d.code, gb, flags, stream);
        else
            rc = p_fused_recurrent_fwd(q.ptr(), k.ptr(), v.ptr(), g.ptr(), beta.ptr(), (const float*)gk.ptr(), nullptr, (const float*)A_log.ptr(),
                                       (const float*)dt_bias.ptr(), (const float*)h0.ptr(), pht, o.data_ptr(), cu.ptr(), slots.ptr(), nullptr, 1,
                                       d.B, d.T, d.H, d.HV, d.K, d.V, N, scale, d.code, gb, flags, stream);
    }
    if (rc != GDN_OK) Py_RETURN_NONE;               // (refused before any launch: the Python path raises)
    return pair(o, ht);
    END_HANDLE_TH_ERRORS
}

// ---- chunked forward ----
// (q, k, v, g, beta, scale, initial_state, output_final_state, state_v_first, cu_seqlens, chunk_indices, scan_tables, A_log, dt_bias,
//  flags); chunk_indices, scan_tables: the tables of checked boundaries, in cu_seqlens' type
struct ChunkArgs {
    Arg q{Py_None}, k{Py_None}, v{Py_None}, g{Py_None}, beta{Py_None}, h0{Py_None}, cu{Py_None}, table{Py_None}, offsets{Py_None}, A_log{Py_None}, dt_bias{Py_None};
    Dims d;
    float scale;
    int gb;
    int64_t N, num_chunks, rows, cols;
    uint32_t flags;
};
// false: not a call for the native path (or an error is set)
bool chunk_args(PyObject* const* a, ChunkArgs& x) {
    x.q = Arg(a[0]); x.k = Arg(a[1]); x.v = Arg(a[2]); x.g = Arg(a[3]); x.beta = Arg(a[4]); x.h0 = Arg(a[6]); x.cu = Arg(a[9]); x.table = Arg(a[10]);
    x.offsets = Arg(a[11]); x.A_log = Arg(a[12]); x.dt_bias = Arg(a[13]);
    const Arg &q = x.q, &k = x.k, &v = x.v, &g = x.g, &beta = x.beta, &h0 = x.h0, &cu = x.cu, &table = x.table, &offsets = x.offsets, &A_log = x.A_log, &dt_bias = x.dt_bias;
    Dims& d = x.d;
    const bool vfirst = truth(a[8]);
    if (!operands(q, k, v, d) || d.code == GDN_DTYPE_F32 || !scale_of(a[5], d.K, x.scale)) return false;
    for (const Arg* t : {&g, &beta, &h0, &cu, &table, &offsets, &A_log, &dt_bias})
        if (!plain(*t, d.dev)) return false;
    if (d.K % 8 || d.V % 8 || d.K > 256 || (d.K <= 128 && d.V > 128) || !beta || !per_head(g, d) || !per_head(beta, d) || !indices(cu, -1)) return false;
    if (!aligned16(q.ptr()) || !aligned16(k.ptr()) || !aligned16(v.ptr()) || !floats(A_log, d.HV) || !floats(dt_bias, d.HV)) return false;
    if ((A_log && !g) || (dt_bias && !A_log)) return false;
    x.gb = gb_code_of(g, beta);
    if (x.gb < 0) return false;
    x.N = cu ? cu->numel() - 1 : d.B;
    if (x.N < 1 || (cu && (d.B != 1 || !table || !offsets || table->dim() != 2 || table->scalar_type() != cu->scalar_type() ||
                           offsets->scalar_type() != cu->scalar_type() || offsets->numel() != 2 * x.N + 1)))
        return false;
    x.num_chunks = cu ? table->size(0) : d.B * ((d.T + 63) / 64);
    x.rows = vfirst ? d.V : d.K; x.cols = vfirst ? d.K : d.V;
    if (h0 && (h0->scalar_type() != at::kFloat || h0->dim() != 4 || h0->size(0) != x.N || h0->size(1) != d.HV || h0->size(2) != x.rows ||
               h0->size(3) != x.cols || !aligned16(h0.ptr())))
        return false;
    x.flags = (uint32_t)PyLong_AsUnsignedLong(a[14]);
    if (PyErr_Occurred()) return false;
    if (vfirst) x.flags |= GDN_FLAG_STATE_V_FIRST;
    if (cu) x.flags |= GDN_FLAG_SEQ_ORDER | (cu->scalar_type() == at::kInt ? GDN_FLAG_CU_INT32 : 0);
    return true;
}
PyObject* chunk_fwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 15) { PyErr_SetString(PyExc_TypeError, "gdn_host.chunk_fwd takes 15 arguments"); return nullptr; }
    ChunkArgs x;
    if (!chunk_args(a, x)) { if (PyErr_Occurred()) return nullptr; Py_RETURN_NONE; }
    const Dims& d = x.d;
    const size_t ws_bytes = p_chunk_workspace_bytes(x.N, d.T, x.num_chunks, d.H, d.HV, d.K, d.V, x.cu ? 1 : 0, x.flags);
    if (ws_bytes == 0) Py_RETURN_NONE;
    const at::Tensor o = empty_on(d.dev, x.v->scalar_type(), x.v->sizes());
    at::Tensor ht;
    if (truth(a[7])) ht = empty_on(d.dev, at::kFloat, {x.N, d.HV, x.rows, x.cols});
    const at::Tensor ws = empty_on(d.dev, at::kByte, {(int64_t)ws_bytes});
    void* stream = stream_of(d.dev);
    int rc;
    {
        const NoGil free;
        rc = p_chunk_fwd(x.q.ptr(), x.k.ptr(), x.v.ptr(), x.g.ptr(), x.beta.ptr(), (const float*)x.A_log.ptr(), (const float*)x.dt_bias.ptr(), (const float*)x.h0.ptr(),
                         ht.defined() ? (float*)ht.data_ptr() : nullptr, o.data_ptr(), x.cu.ptr(), x.table.ptr(), x.offsets.ptr(), ws.data_ptr(), ws_bytes,
                         d.B, d.T, d.H, d.HV, d.K, d.V, x.N, x.num_chunks, x.scale, d.code, x.gb, x.flags, stream);
    }
    if (rc != GDN_OK) Py_RETURN_NONE;
    return pair(o, ht);
    END_HANDLE_TH_ERRORS
}

// ---- one decode step of the layer ----
// (x [N,1,hidden], q, k, v, a, b, g, o weights, A_log, dt_bias, (q, k, v conv weights [D,1,W]), (q, k, v conv biases), (q, k, v conv
//  states [N,D,W]), recurrent state [N,HV,V,K], norm weight, norm eps, neg_eigval, num_heads): four launches - the six projections
// with the convolutions' update and the gate's and beta's activations, the recurrence on the state where it is, the gated norm, the
// output projection.  The states are updated in place.
PyObject* layer_step(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 18) { PyErr_SetString(PyExc_TypeError, "gdn_host.layer_step takes 18 arguments"); return nullptr; }
    const Arg x(a[0]), qw(a[1]), kw(a[2]), vw(a[3]), aw(a[4]), bw(a[5]), gw(a[6]), ow(a[7]), A_log(a[8]), dt_bias(a[9]), state(a[13]), norm_w(a[14]);
    if (!x || !x->is_cuda() || x->dim() != 3 || x->size(1) != 1) Py_RETURN_NONE;
    const c10::Device dev = x->device();
    const at::ScalarType type = x->scalar_type();
    const int code = code_of(type);
    if ((code != GDN_DTYPE_BF16 && code != GDN_DTYPE_F16) || dev.index() != c10::hip::current_device()) Py_RETURN_NONE;
    const int64_t N = x->size(0), hidden = x->size(2), H = PyLong_AsLongLong(a[17]);
    if (PyErr_Occurred()) return nullptr;
    for (const Arg* t : {&x, &qw, &kw, &vw, &aw, &bw, &gw, &ow, &A_log, &dt_bias, &state, &norm_w})
        if (!*t || !plain(*t, dev) || !aligned16(t->ptr())) Py_RETURN_NONE;
    for (const Arg* t : {&qw, &kw, &vw, &aw, &bw, &gw})
        if (t->t->scalar_type() != type || t->t->dim() != 2 || t->t->size(1) != hidden) Py_RETURN_NONE;
    if (state->scalar_type() != at::kFloat || state->dim() != 4 || state->size(0) != N) Py_RETURN_NONE;
    const int64_t HV = state->size(1), V = state->size(2), K = state->size(3), kd = H * K, vd = HV * V;
    if (N < 1 || H < 1 || HV % H || K % 4 || V % 8 || K > 256 || hidden % 256 || vd % 256 || qw->size(0) != kd || kw->size(0) != kd || vw->size(0) != vd ||
        gw->size(0) != vd || aw->size(0) != HV || bw->size(0) != HV || ow->scalar_type() != type || ow->dim() != 2 || ow->size(1) != vd ||
        A_log->numel() != HV || dt_bias->numel() != HV || A_log->scalar_type() != dt_bias->scalar_type() || norm_w->numel() != V)
        Py_RETURN_NONE;
    const int gate_code = code_of(A_log->scalar_type()), norm_code = code_of(norm_w->scalar_type());
    if (gate_code < 0 || norm_code < 0) Py_RETURN_NONE;
    const int64_t out_cols = ow->size(0);
    // Many sequences of a large layer leave the host time behind and are products of a library's size: there the modules are faster.
    // Native and by modules, us a step: 6 heads of 256 x 512 at 2048 (25.2 M weights), 129 sequences 219 and 335, 192 296 and 334, 256 376
    // and 369, 512 701 and 666; 8 heads of 128 at 1024 (5.3 M weights), 129 sequences 61 and 325, 512 147 and 325, 1024 260 and 327.
    if (N > 128 && N * ((2 * kd + 2 * vd + 2 * HV) * hidden + vd * out_cols) > 5600000000ll) Py_RETURN_NONE;
    // Every limit of the four launches: none may be refused once the first has moved the convolutions' states on.
    if (N > GDN_STEP_MAX_ROWS || std::max({hidden, kd, vd, out_cols}) > GDN_STEP_MAX_COLS || out_cols < 1 || V > GDN_NORM_MAX_ROW_BYTES / 2 ||
        (N + 8) * HV * ((V + 31) / 32) >= (1ll << 31))
        Py_RETURN_NONE;
    gdn_step_segment seg[6] = {};
    for (int i = 10; i < 13; ++i)
        if (!PyTuple_Check(a[i]) || PyTuple_GET_SIZE(a[i]) != 3) Py_RETURN_NONE;
    for (int i = 0; i < 3; ++i) {
        const Arg w(PyTuple_GetItem(a[10], i)), bias(PyTuple_GetItem(a[11], i)), st(PyTuple_GetItem(a[12], i));
        const int64_t D = i < 2 ? kd : vd;
        if (!w || !st || !plain(w, dev) || !plain(bias, dev) || !plain(st, dev) || w->scalar_type() != type || st->scalar_type() != type) Py_RETURN_NONE;
        const int64_t W = w->size(-1);
        if (W < 1 || W > 8 || w->numel() != D * W || st->dim() != 3 || st->size(0) != N || st->size(1) != D || st->size(2) != W ||
            (bias && (bias->scalar_type() != type || bias->numel() != D)) || !aligned16(w.ptr()) || !aligned16(st.ptr()))
            Py_RETURN_NONE;
        const Arg& pw = i == 0 ? qw : i == 1 ? kw : vw;
        seg[i] = {pw.ptr(), D, nullptr, w.ptr(), bias.ptr(), st.ptr(), nullptr, nullptr, GDN_STEP_CONV, (int)W, 0, 0};
    }
    seg[3] = {gw.ptr(), vd, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, GDN_STEP_PLAIN, 0, 0, 0};
    seg[4] = {aw.ptr(), HV, nullptr, nullptr, nullptr, nullptr, A_log.ptr(), dt_bias.ptr(), GDN_STEP_GATE, 0, gate_code, 0};
    seg[5] = {bw.ptr(), HV, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, truth(a[16]) ? GDN_STEP_BETA2 : GDN_STEP_BETA, 0, 0, 0};
    const float eps = (float)PyFloat_AsDouble(a[15]);
    if (PyErr_Occurred()) return nullptr;
    const at::Tensor out = empty_on(dev, type, {N, 1, out_cols});
    // one allocation for everything in between, each part 256-byte aligned
    int64_t at_byte = 0;
    auto take = [&](int64_t bytes) { const int64_t at = at_byte; at_byte += (bytes + 255) / 256 * 256; return at; };
    const int64_t o_q = take(N * kd * 2), o_k = take(N * kd * 2), o_v = take(N * vd * 2), o_gate = take(N * vd * 2), o_o = take(N * vd * 2),
                  o_y = take(N * vd * 2), o_g = take(N * HV * 4), o_b = take(N * HV * 4);
    const at::Tensor ws = empty_on(dev, at::kByte, {at_byte});
    char* base = (char*)ws.data_ptr();
    seg[0].out = base + o_q; seg[1].out = base + o_k; seg[2].out = base + o_v; seg[3].out = base + o_gate; seg[4].out = base + o_g; seg[5].out = base + o_b;
    gdn_step_segment last = {};
    last.weight = ow.ptr(); last.cols = out_cols; last.out = out.data_ptr(); last.kind = GDN_STEP_PLAIN;
    void* stream = stream_of(dev);
    int rc;
    {
        const NoGil free;
        rc = p_step_linear(x.ptr(), N, hidden, seg, 6, code, stream);
        if (rc == GDN_OK)
            rc = p_fused_recurrent_fwd(base + o_q, base + o_k, base + o_v, base + o_g, base + o_b, nullptr, nullptr, nullptr, nullptr, (const float*)state.ptr(),
                                       (float*)state.ptr(), base + o_o, nullptr, nullptr, nullptr, 1, N, 1, H, HV, K, V, N, (float)std::pow((double)K, -0.5), code,
                                       GDN_DTYPE_F32, GDN_FLAG_QK_L2NORM | GDN_FLAG_STATE_V_FIRST, stream);
        if (rc == GDN_OK)
            rc = p_norm_gated_fwd(base + o_o, base + o_gate, norm_w.ptr(), nullptr, nullptr, base + o_y, nullptr, nullptr, nullptr, N * HV, V, eps, code, norm_code,
                                  GDN_DTYPE_F32, GDN_DTYPE_F32, GDN_ACT_SILU, 1, stream);
        if (rc == GDN_OK) rc = p_step_linear(base + o_y, N, vd, &last, 1, code, stream);
    }
    check_rc(rc, "gdn_host.layer_step");
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

#include "gdn_host_train.h"

PyMethodDef methods[] = {
    {"chunk_train", (PyCFunction)(void*)chunk_train, METH_FASTCALL, "chunked operator with gradients; None: not a call for the native path"},
    {"layer_train", (PyCFunction)(void*)layer_train, METH_FASTCALL, "the layer's forward with gradients; None: not a call for the native path"},
    {"layer_step", (PyCFunction)(void*)layer_step, METH_FASTCALL, "one decode step of the layer; None: not a call for the native path"},
    {"bind", bind, METH_O, "bind({name: address}) - entry points of libgdn_hip.so"},
    {"fused_recurrent", (PyCFunction)(void*)fused_recurrent, METH_FASTCALL, "token recurrence; None: not a call for the native path"},
    {"chunk_fwd", (PyCFunction)(void*)chunk_fwd, METH_FASTCALL, "chunked forward; None: not a call for the native path"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "gdn_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// (the extension holds for the torch it was built with; the binding looks)
PyMODINIT_FUNC PyInit_gdn_host() {
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "TORCH_VERSION", GDN_TORCH_VERSION) < 0) { Py_DECREF(m); return nullptr; }
    return m;
}
