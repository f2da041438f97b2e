// The host path between Python and the C ABI of libflame_attn_hip.so, as a CPython extension on torch's C++ API:
// argument unpacking, output and workspace allocation, the autograd node of the scaled dot-product attention, and the
// call itself.  No arithmetic and no fallback: every function ends in one or two calls of the C ABI.
//
// Why it is native: the small calls are bound by the host, not by their kernels.  Through ctypes and a Python
// torch.autograd.Function one training step of [1, 4, 256, 64] kept the host busy for 88 us for 29 us of kernels (and a
// forward alone for 20 us): argument objects, four stride arrays per tensor, and a backward that had to take the
// interpreter lock on autograd's device thread.
//
// The library is not linked: bind() receives the handle that the Python side opened (so that an override of the library
// path holds here as well) and looks the entry points up in it.
#include <Python.h>

#include <dlfcn.h>

#include <algorithm>
#include <cmath>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>      // this torch names its HIP devices "cuda"
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "../../include/flame_attn.h"
#include "mask_route.hpp"

namespace {

using at::Tensor;

#define FLAME_HOST_ENTRY_POINTS(X)                                                                                      \
    X(flame_attn_fwd_bf16) X(flame_attn_fwd_ws_bf16) X(flame_attn_fwd_workspace_bytes) X(flame_attn_fwd_scratch_bytes) X(flame_attn_mask_workspace_bytes) \
    X(flame_attn_fwd_bias_bf16)                                                                                         \
    X(flame_attn_bwd_bf16) X(flame_attn_bwd_workspace_bytes) X(flame_attn_fwd_dropout_tiled_bf16)                       \
    X(flame_attn_bwd_dropout_tiled_bf16) X(flame_attn_materialised_workspace_bytes) X(flame_attn_fwd_materialised_bf16) \
    X(flame_attn_bwd_materialised_bf16) X(flame_sage_quant_qk_int8_ks) X(flame_sage_attn_fwd_bias_int8)                 \
    X(flame_attn_prep_rmsnorm_rope_bf16) X(flame_bf16_to_fp8) X(flame_fp8_to_bf16) X(flame_attn_cast_qkv_f32_to_bf16) X(flame_attn_cast_bf16_to_f32)

struct Api {
#define FLAME_HOST_MEMBER(name) decltype(&::name) name = nullptr;
    FLAME_HOST_ENTRY_POINTS(FLAME_HOST_MEMBER)
#undef FLAME_HOST_MEMBER
};
Api g_api;
PyObject* g_error_class = nullptr;      // FlameAttnError(fn, code)

// ---------------------------------------------------------------- errors
struct CallError {                      // a C ABI call that returned non-zero
    const char* fn;
    int code;
};
struct PyErrorSet {};                   // a Python exception is set already

void set_python_error(const CallError& e) {
    PyObject* obj = PyObject_CallFunction(g_error_class, "si", e.fn, e.code);
    if (obj) {
        PyErr_SetObject(g_error_class, obj);
        Py_DECREF(obj);
    }
}
[[noreturn]] void fail(PyObject* type, const char* what) {
    PyErr_SetString(type, what);
    throw PyErrorSet{};
}
void check_that(bool ok, const char* what) {
    if (!ok) fail(PyExc_AssertionError, what);
}
void check_rc(int rc, const char* fn) {
    if (rc != FLAME_ATTN_OK) throw CallError{fn, rc};
}
template <class F>
PyObject* guarded(F&& f) {
    HANDLE_TH_ERRORS
    // torch.jit.trace records torch's operators only: the results of these calls would become constants of the trace
    TORCH_CHECK(!torch::jit::tracer::isTracing(), "the attention calls cannot be recorded by torch.jit.trace");
    try {
        return f();
    } catch (const CallError& e) {
        set_python_error(e);
        return nullptr;
    } catch (const PyErrorSet&) {
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}
struct WithoutGil {
    PyThreadState* state = PyEval_SaveThread();
    ~WithoutGil() { PyEval_RestoreThread(state); }
};

// ---------------------------------------------------------------- arguments
const Tensor& tensor_arg(PyObject* o, const char* what) {
    if (!THPVariable_Check(o)) fail(PyExc_TypeError, what);
    return THPVariable_Unpack(o);
}
Tensor opt_tensor_arg(PyObject* o, const char* what) { return o == Py_None ? Tensor() : tensor_arg(o, what); }
double float_arg(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw PyErrorSet{};
    return v;
}
long long_arg(PyObject* o) {
    const long v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) throw PyErrorSet{};
    return v;
}
uint64_t u64_arg(PyObject* o) {         // the low 64 bits
    const uint64_t v = PyLong_AsUnsignedLongLongMask(o);
    if (PyErr_Occurred()) throw PyErrorSet{};
    return v;
}
bool bool_arg(PyObject* o) {
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw PyErrorSet{};
    return v != 0;
}
void need_args(Py_ssize_t got, Py_ssize_t want) {
    if (got != want) fail(PyExc_TypeError, "wrong number of arguments");
}

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
const int64_t* strides4(const Tensor& t) { return t.strides().data(); }
void check_4d(const Tensor& t) {
    if (t.dim() != 4) fail(PyExc_ValueError, "expected a 4-D tensor");
}
struct Sizes {
    int B, H, Sq, Sk, D;
};
Sizes sizes_of(const Tensor& q, const Tensor& k) {
    check_4d(q);
    check_4d(k);
    return {(int)q.size(0), (int)q.size(1), (int)q.size(2), (int)k.size(2), (int)q.size(3)};
}

// Element strides of a [B|1, H|1, Sq|1, Sk|1] tensor over the full index space (0 broadcasts); false: not broadcastable.
bool broadcast_strides(const Tensor& m, const Sizes& z, int64_t (&st)[4]) {
    const int64_t full[4] = {z.B, z.H, z.Sq, z.Sk};
    if (m.dim() != 4) return false;
    for (int ax = 0; ax < 4; ++ax) {
        const int64_t n = m.size(ax);
        if (n != 1 && n != full[ax]) return false;
        st[ax] = (n == 1 && full[ax] != 1) ? 0 : m.stride(ax);
    }
    return true;
}
struct MaskView {
    const uint8_t* data = nullptr;
    int64_t st[4] = {0, 0, 0, 0};
    const int64_t* strides() const { return data ? st : nullptr; }
};
MaskView mask_view(const Tensor& m, const Sizes& z) {
    MaskView v;
    if (!m.defined()) return v;
    check_that(m.scalar_type() == at::kByte && m.dim() == 4, "the mask is a 4-D uint8 tensor");
    check_that(broadcast_strides(m, z, v.st), "mask is not broadcastable to [B,H,Sq,Sk]");
    v.data = static_cast<const uint8_t*>(m.data_ptr());
    return v;
}
struct BiasView {
    const void* data = nullptr;
    int dtype = FLAME_ATTN_DTYPE_F32;
    int64_t st[4] = {0, 0, 0, 0};
    const int64_t* strides() const { return data ? st : nullptr; }
};
BiasView bias_view(const Tensor& b, const Sizes& z) {
    BiasView v;
    if (!b.defined()) return v;
    check_that(b.dim() == 4 && (b.scalar_type() == at::kFloat || b.scalar_type() == at::kBFloat16), "the bias is a 4-D fp32 or bf16 tensor");
    check_that(broadcast_strides(b, z, v.st), "bias is not broadcastable to [B,H,Sq,Sk]");
    v.dtype = b.scalar_type() == at::kFloat ? FLAME_ATTN_DTYPE_F32 : FLAME_ATTN_DTYPE_BF16;
    v.data = b.data_ptr();
    return v;
}

Tensor empty(at::IntArrayRef size, at::ScalarType dt, const Tensor& like) {
    return at::Tensor(at::detail::empty_cuda(size, dt, like.device(), std::nullopt));
}
Tensor bytes_like(size_t n, const Tensor& like) { return empty({(int64_t)n}, at::kByte, like); }
// Room that a call is faster with but does not need (up to 1 GiB of mask words, one slice's probabilities): undefined where the
// device has none left.
Tensor optional_bytes_like(size_t n, const Tensor& like) {
    if (n == 0) return Tensor();
    try {
        return bytes_like(n, like);
    } catch (const c10::OutOfMemoryError&) {
        return Tensor();
    }
}
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream(); }

// ---------------------------------------------------------------- forward and backward
// Room that a mask as bits takes; none for calls that would not form them, nor for head dims that the fused kernels refuse with a
// mask, which go on to the materialised path.
size_t mask_room(const Sizes& z, const MaskView& mask, const Tensor& kv_len, bool causal, bool backward) {
    if (!mask.data || z.D > 128 || z.D % 8 != 0) return 0;
    const bool rows16 = fattn::mask_rows16(mask.data, mask.st[0], mask.st[1], mask.st[2], mask.st[3]);
    if (!fattn::mask_bits_pay(backward, rows16, mask.st[1] != 0 && z.H > 1, mask.st[2], z.Sq, z.Sk, causal)) return 0;
    return g_api.flame_attn_mask_workspace_bytes(z.B, z.H, z.Sq, z.Sk, mask.strides(), kv_len.defined(), causal);
}
struct FwdOpts {
    bool causal = false;
    Tensor kv_len, workspace;
    MaskView mask;
    bool want_lse = true;
};

// rc of the call; o and lse are allocated where they are not given
int call_fwd(const Tensor& q, const Tensor& k, const Tensor& v, const Sizes& z, float scale, const FwdOpts& f, Tensor& o, Tensor& lse) {
    if (!o.defined()) o = empty({z.B, z.H, z.Sq, z.D}, at::kBFloat16, q);
    if (!lse.defined() && f.want_lse) lse = empty({(int64_t)z.B * z.H, z.Sq}, at::kFloat, q);
    Tensor ws = f.workspace;
    if (!ws.defined()) {       // room for the slices of a key split, where the grid would leave compute units idle, or for the mask as bits
        const size_t need = f.mask.data ? mask_room(z, f.mask, f.kv_len, f.causal, false) : g_api.flame_attn_fwd_scratch_bytes(z.B, z.H, z.Sq, z.Sk, z.D);
        ws = optional_bytes_like(need, q);
        if (need && !ws.defined() && !f.mask.data) {       // the probabilities of wide heads do not fit: partial outputs may
            const size_t less = g_api.flame_attn_fwd_workspace_bytes(z.B, z.H, z.Sq, z.Sk, z.D);
            if (less < need) ws = optional_bytes_like(less, q);
        }
    }
    if (ws.defined())
        return g_api.flame_attn_fwd_ws_bf16(ptr(q), ptr(k), ptr(v), ptr(o), ptr(lse), z.B, z.H, z.Sq, z.Sk, z.D, scale, strides4(q), strides4(k),
                                            strides4(v), strides4(o), 0, 0, 0, 0, 0, f.causal, static_cast<const int32_t*>(ptr(f.kv_len)), f.mask.data,
                                            f.mask.strides(), ptr(ws), (size_t)ws.numel(), stream_of(q));
    return g_api.flame_attn_fwd_bf16(ptr(q), ptr(k), ptr(v), ptr(o), ptr(lse), z.B, z.H, z.Sq, z.Sk, z.D, scale, strides4(q), strides4(k),
                                     strides4(v), strides4(o), 0, 0, 0, 0, 0, f.causal, static_cast<const int32_t*>(ptr(f.kv_len)), f.mask.data,
                                     f.mask.strides(), stream_of(q));
}

struct Grads {
    Tensor dq, dk, dv;
};
void alloc_grads(const Tensor& q, const Sizes& z, Grads& g) {
    g.dq = empty({z.B, z.H, z.Sq, z.D}, at::kBFloat16, q);
    g.dk = empty({z.B, z.H, z.Sk, z.D}, at::kBFloat16, q);
    g.dv = empty({z.B, z.H, z.Sk, z.D}, at::kBFloat16, q);
}
int call_bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& d_o, const Tensor& lse, const Sizes& z, float scale,
             bool causal, const Tensor& kv_len, const MaskView& mask, Tensor workspace, Grads& g) {
    if (!workspace.defined()) {
        const size_t need = g_api.flame_attn_bwd_workspace_bytes(z.B, z.H, z.Sq, z.D);
        const size_t words = mask_room(z, mask, kv_len, causal, true);
        if (words) workspace = optional_bytes_like(need + words, q);
        if (!workspace.defined()) workspace = bytes_like(need, q);
    }
    if (!g.dq.defined()) alloc_grads(q, z, g);
    return g_api.flame_attn_bwd_bf16(ptr(q), ptr(k), ptr(v), ptr(o), ptr(d_o), ptr(lse), ptr(g.dq), ptr(g.dk), ptr(g.dv), z.B, z.H, z.Sq, z.Sk, z.D,
                                     scale, strides4(q), strides4(k), strides4(v), strides4(o), strides4(d_o), strides4(g.dq), strides4(g.dk),
                                     strides4(g.dv), 0, 0, 0, 0, 0, 0, 0, 0, 0, causal, static_cast<const int32_t*>(ptr(kv_len)), mask.data,
                                     mask.strides(), ptr(workspace), (size_t)workspace.numel(), stream_of(q));
}

// the materialised path: any head dim (the reference's dispatch, src/sdpa.rs:483-587)
int call_fwd_materialised(const Tensor& q, const Tensor& k, const Tensor& v, const Sizes& z, float scale, bool causal, const MaskView& mask, Tensor& o,
                          Tensor& lse) {
    const int Dv = (int)v.size(3);
    o = empty({z.B, z.H, z.Sq, Dv}, at::kBFloat16, q);
    lse = empty({(int64_t)z.B * z.H, z.Sq}, at::kFloat, q);
    const Tensor ws = bytes_like(g_api.flame_attn_materialised_workspace_bytes(z.B, z.H, z.Sq, z.Sk, z.D, Dv, 0), q);
    return g_api.flame_attn_fwd_materialised_bf16(ptr(q), ptr(k), ptr(v), ptr(o), ptr(lse), z.B, z.H, z.Sq, z.Sk, z.D, Dv, scale, strides4(q), strides4(k),
                                                  strides4(v), strides4(o), 0, 0, 0, 0, 0, causal, nullptr, mask.data, mask.strides(), nullptr,
                                                  FLAME_ATTN_DTYPE_BF16, nullptr, 0.f, 0, 0, 0, ptr(ws), (size_t)ws.numel(), stream_of(q));
}
int call_bwd_materialised(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& d_o, const Tensor& lse, const Sizes& z,
                          float scale, bool causal, const MaskView& mask, Grads& g) {
    const int Dv = (int)v.size(3);
    const Tensor ws = bytes_like(g_api.flame_attn_materialised_workspace_bytes(z.B, z.H, z.Sq, z.Sk, z.D, Dv, 1), q);
    g.dq = at::empty_like(q);
    g.dk = at::empty_like(k);
    g.dv = at::empty_like(v);
    return g_api.flame_attn_bwd_materialised_bf16(ptr(q), ptr(k), ptr(v), ptr(o), ptr(d_o), ptr(lse), ptr(g.dq), ptr(g.dk), ptr(g.dv), z.B, z.H, z.Sq,
                                                  z.Sk, z.D, Dv, scale, strides4(q), strides4(k), strides4(v), strides4(o), strides4(d_o), strides4(g.dq),
                                                  strides4(g.dk), strides4(g.dv), 0, 0, 0, 0, 0, 0, 0, 0, 0, causal, nullptr, mask.data, mask.strides(), 0.f,
                                                  0, 0, 0, ptr(ws), (size_t)ws.numel(), stream_of(q));
}

// ---------------------------------------------------------------- sdpa
// rows that start on 16 bytes, D contiguous: what the kernels load
bool rows_aligned(const Tensor& t) {
    return t.stride(3) == 1 && ((t.stride(0) | t.stride(1) | t.stride(2)) & 7) == 0 && (t.storage_offset() & 7) == 0;
}
Tensor as_bf16_view(const Tensor& x) {
    Tensor t = x.scalar_type() == at::kBFloat16 ? x : x.to(at::kBFloat16);      // promote_bf16 of the reference
    if (t.size(3) % 8 == 0 ? !rows_aligned(t) : t.stride(3) != 1) t = t.contiguous();
    return t;
}

// A tensor whose elements are what its address and strides say, where no subclass, mode or transform, of the tensor's or of the
// calling thread's, has a part in what .to() does to it.
bool plain_f32(const Tensor& t) {
    static const c10::DispatchKeySet special({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::PythonDispatcher,
                                              c10::DispatchKey::Functionalize, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                              c10::DispatchKey::FuncTorchVmapMode, c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
                                              c10::DispatchKey::Batched, c10::DispatchKey::VmapMode, c10::DispatchKey::Conjugate,
                                              c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
    if ((t.key_set() | c10::impl::tls_local_dispatch_key_set().included_).has_any(special)) return false;
    if (t.scalar_type() != at::kFloat || !t.is_cuda() || t.layout() != at::kStrided || t.stride(3) != 1) return false;
    for (int ax = 0; ax < 3; ++ax)          // .to() keeps such strides, and the kernels refuse them
        if (t.size(ax) == 1 && t.stride(ax) % 8 != 0) return false;
    return true;
}
// Where no graph is recorded, fp32 Q, K and V become bf16 in one launch instead of three, and the output fp32 in one: of a small
// call's time most was the four conversions of the tensor library and the gaps between them.  false: not these tensors.
// (Whole call, us: B=2 H=12 S=77 D=64 24 -> 13, B=1 H=16 S=257 D=80 24 -> 14.7, B=2 H=16 S=577 D=64 24 -> 21.7.  Large ones gain
// nothing: 19 million elements in Q, K and V 86.7 -> 87.3, 25 million 178 -> 181.)
constexpr int64_t kMostCast = (int64_t)12 << 20;
bool cast_qkv(const Tensor& q, const Tensor& k, const Tensor& v, Tensor& qb, Tensor& kb, Tensor& vb) {
    if (!plain_f32(q) || !plain_f32(k) || !plain_f32(v)) return false;
    if (k.device() != q.device() || v.device() != q.device() || k.sizes() != v.sizes() || q.size(0) != k.size(0) || q.size(1) != k.size(1) ||
        q.size(3) != k.size(3) || q.size(3) % 8 != 0 || q.numel() == 0 || k.numel() == 0 || q.numel() + 2 * k.numel() > kMostCast)
        return false;
    for (int64_t n : q.sizes())
        if (n > INT32_MAX) return false;
    if (k.size(2) > INT32_MAX) return false;
    qb = empty(q.sizes(), at::kBFloat16, q);
    kb = empty(k.sizes(), at::kBFloat16, q);
    vb = empty(v.sizes(), at::kBFloat16, q);
    return g_api.flame_attn_cast_qkv_f32_to_bf16(ptr(q), ptr(k), ptr(v), ptr(qb), ptr(kb), ptr(vb), (int)q.size(0), (int)q.size(1), (int)q.size(2),
                                                 (int)k.size(2), (int)q.size(3), strides4(q), strides4(k), strides4(v), stream_of(q)) == FLAME_ATTN_OK;
}
Tensor f32_of(const Tensor& o) {       // contiguous bf16
    Tensor out = empty(o.sizes(), at::kFloat, o);
    check_rc(g_api.flame_attn_cast_bf16_to_f32(ptr(o), ptr(out), o.numel(), stream_of(o)), "flame_attn_cast_bf16_to_f32");
    return out;
}

// The copy of a keep-mask that a recorded graph holds, so that the caller may refill the buffer before the backward.  Axes
// along which the tensor repeats itself are kept once, and rows start on 16 bytes (where the kernels load them as vectors).
// One launch: 3 us of a training step of 185 us (B=4 H=16 S=1101 D=128, a mask of keys).
Tensor own_mask(const Tensor& m) {
    Tensor src = m;
    for (int ax = 0; ax < 4; ++ax)
        if (src.stride(ax) == 0 && src.size(ax) > 1) src = src.narrow(ax, 0, 1);
    const int64_t n = src.size(3);
    Tensor own = empty({src.size(0), src.size(1), src.size(2), (n + 15) / 16 * 16}, at::kBool, m).narrow(3, 0, n);
    at::ne_out(own, src, 0);
    return own.view(at::kByte);
}

// forward of one call; true: served by the materialised path
bool sdpa_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& mask, bool causal, double scale, bool want_lse, Tensor& o, Tensor& lse) {
    const Sizes z{(int)q.size(0), (int)q.size(1), (int)q.size(2), (int)k.size(2), (int)q.size(3)};
    FwdOpts f;
    f.causal = causal;
    f.want_lse = want_lse;
    if (mask.defined()) {
        broadcast_strides(mask, z, f.mask.st);          // checked by the caller
        f.mask.data = static_cast<const uint8_t*>(mask.data_ptr());
    }
    int rc = call_fwd(q, k, v, z, (float)scale, f, o, lse);
    if (rc == FLAME_ATTN_OK) return false;
    if (rc != FLAME_ATTN_ERR_UNSUPPORTED) throw CallError{"flame_attn_fwd_bf16", rc};
    rc = call_fwd_materialised(q, k, v, z, (float)scale, causal, f.mask, o, lse);
    check_rc(rc, "flame_attn_fwd_materialised_bf16");
    return true;
}

// A failed call on autograd's thread becomes the same Python exception there.
[[noreturn]] void throw_python(const CallError& e) {
    PyGILState_STATE g = PyGILState_Ensure();
    set_python_error(e);
    python_error err;
    err.persist();
    PyGILState_Release(g);
    throw err;
}

struct Sdpa : public torch::autograd::Function<Sdpa> {
    // saves O and the log-sum-exp only; the backward recomputes the probabilities
    static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const std::optional<Tensor>& mask,
                          bool causal, double scale) {
        Tensor o, lse;
        const Tensor m = mask.has_value() ? *mask : Tensor();
        const bool materialised = sdpa_forward(q, k, v, m, causal, scale, true, o, lse);
        ctx->save_for_backward({q, k, v, o, lse, m});
        ctx->saved_data["causal"] = causal;
        ctx->saved_data["scale"] = scale;
        ctx->saved_data["materialised"] = materialised;
        return o;
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &o = saved[3], &lse = saved[4], &m = saved[5];
        const bool causal = ctx->saved_data["causal"].toBool();
        const float scale = (float)ctx->saved_data["scale"].toDouble();
        c10::OptionalDeviceGuard device(q.device());
        at::NoGradGuard no_grad;
        const Sizes z{(int)q.size(0), (int)q.size(1), (int)q.size(2), (int)k.size(2), (int)q.size(3)};
        Tensor d_o = grads[0].to(at::kBFloat16);
        if (d_o.stride(3) != 1 || ((d_o.stride(0) | d_o.stride(1) | d_o.stride(2)) & 7) != 0) d_o = d_o.contiguous();
        MaskView mv;
        if (m.defined()) {
            broadcast_strides(m, z, mv.st);
            mv.data = static_cast<const uint8_t*>(m.data_ptr());
        }
        Grads g;
        int rc = FLAME_ATTN_ERR_UNSUPPORTED;
        if (!ctx->saved_data["materialised"].toBool() && z.D <= 128) rc = call_bwd(q, k, v, o, d_o, lse, z, scale, causal, Tensor(), mv, Tensor(), g);
        if (rc == FLAME_ATTN_ERR_UNSUPPORTED) {         // a head dim the fused forward serves and the fused backward does not
            rc = call_bwd_materialised(q, k, v, o, d_o, lse, z, scale, causal, mv, g);
            if (rc != FLAME_ATTN_OK) throw_python({"flame_attn_bwd_materialised_bf16", rc});
        } else if (rc != FLAME_ATTN_OK) {
            throw_python({"flame_attn_bwd_bf16", rc});
        }
        return {g.dq, g.dk, g.dv, Tensor(), Tensor(), Tensor()};
    }
};

// sdpa(q, k, v, mask | None, causal, scale | None)
PyObject* py_sdpa(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need_args(n, 6);
        const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v");
        if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4) fail(PyExc_ValueError, "SDPA expects 4-D input [B, H, S, D]");
        // whether or not a graph is recorded: without one the autograd node, which has no jvp either, is passed by
        for (const Tensor* t : {&q, &k, &v})
            TORCH_CHECK_NOT_IMPLEMENTED(!t->_fw_grad(0).defined(), "SDPA has no forward-mode derivative: an input carries a tangent");
        const bool causal = bool_arg(a[4]);
        const double scale = a[5] == Py_None ? 1.0 / std::sqrt((double)q.size(3)) : float_arg(a[5]);
        Tensor mask;
        bool converted = false;      // the mask is a tensor of its own already
        if (!causal && a[3] != Py_None) {
            const Tensor& m = tensor_arg(a[3], "attn_mask");
            if (m.dim() != 4) fail(PyExc_ValueError, "mask must be 4D [B,H,Q,K]");
            // a boolean tensor holds one byte of 0 or 1 per element already
            converted = m.scalar_type() != at::kByte && m.scalar_type() != at::kBool;
            mask = m.scalar_type() == at::kByte ? m : (converted ? m.to(at::kFloat).ge(0.5) : m).view(at::kByte);
            int64_t st[4];
            const Sizes z{(int)q.size(0), (int)q.size(1), (int)q.size(2), (int)k.size(2), (int)q.size(3)};
            check_that(broadcast_strides(mask, z, st), "mask is not broadcastable to [B,H,Sq,Sk]");
        }
        Tensor out;
        {
            WithoutGil nogil;
            c10::OptionalDeviceGuard device(q.device());
            const at::ScalarType orig = q.scalar_type();
            Tensor qb, kb, vb, lse;
            const bool graph = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad());
            if (!graph && cast_qkv(q, k, v, qb, kb, vb)) {
                sdpa_forward(qb, kb, vb, mask, causal, scale, false, out, lse);
                out = f32_of(out);
            } else if (qb = as_bf16_view(q), kb = as_bf16_view(k), vb = as_bf16_view(v);
                       at::GradMode::is_enabled() && (qb.requires_grad() || kb.requires_grad() || vb.requires_grad())) {
                out = Sdpa::apply(qb, kb, vb, mask.defined() ? std::optional<Tensor>(converted ? mask : own_mask(mask)) : std::nullopt, causal, scale);
            } else {
                sdpa_forward(qb, kb, vb, mask, causal, scale, false, out, lse);
            }
            if (orig != at::kBFloat16) out = out.to(orig);
        }
        return THPVariable_Wrap(out);
    });
}

PyObject* pair(const Tensor& a, const Tensor& b) {
    PyObject* pa = THPVariable_Wrap(a);
    PyObject* pb = b.defined() ? THPVariable_Wrap(b) : Py_NewRef(Py_None);
    PyObject* t = PyTuple_Pack(2, pa, pb);
    Py_DECREF(pa);
    Py_DECREF(pb);
    return t;
}
PyObject* triple(const Grads& g) {
    PyObject* p[3] = {THPVariable_Wrap(g.dq), THPVariable_Wrap(g.dk), THPVariable_Wrap(g.dv)};
    PyObject* t = PyTuple_Pack(3, p[0], p[1], p[2]);
    for (PyObject* x : p) Py_DECREF(x);
    return t;
}

// attn_fwd(q, k, v, scale, causal, kv_len, mask, want_lse, out, lse_out, workspace) -> (o, lse | None)
PyObject* py_attn_fwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need_args(n, 11);
        const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v");
        const Sizes z = sizes_of(q, k);
        check_4d(v);
        FwdOpts f;
        const float scale = (float)float_arg(a[3]);
        f.causal = bool_arg(a[4]);
        f.kv_len = opt_tensor_arg(a[5], "kv_len");
        f.mask = mask_view(opt_tensor_arg(a[6], "mask"), z);
        f.want_lse = bool_arg(a[7]);
        Tensor o = opt_tensor_arg(a[8], "out"), lse = opt_tensor_arg(a[9], "lse_out");
        f.workspace = opt_tensor_arg(a[10], "workspace");
        {
            WithoutGil nogil;
            c10::OptionalDeviceGuard device(q.device());
            check_rc(call_fwd(q, k, v, z, scale, f, o, lse), f.workspace.defined() ? "flame_attn_fwd_ws_bf16" : "flame_attn_fwd_bf16");
        }
        return pair(o, lse);
    });
}

// attn_bwd(q, k, v, o, do, lse, scale, causal, kv_len, mask, workspace, dq, dk, dv) -> (dq, dk, dv)
PyObject* py_attn_bwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need_args(n, 14);
        const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v"), &o = tensor_arg(a[3], "o"),
                     &d_o = tensor_arg(a[4], "do"), &lse = tensor_arg(a[5], "lse");
        const Sizes z = sizes_of(q, k);
        check_4d(v), check_4d(o), check_4d(d_o);
        const float scale = (float)float_arg(a[6]);
        const bool causal = bool_arg(a[7]);
        const Tensor kv_len = opt_tensor_arg(a[8], "kv_len");
        const MaskView mask = mask_view(opt_tensor_arg(a[9], "mask"), z);
        const Tensor ws = opt_tensor_arg(a[10], "workspace");
        Grads g{opt_tensor_arg(a[11], "dq"), opt_tensor_arg(a[12], "dk"), opt_tensor_arg(a[13], "dv")};
        if (g.dq.defined()) check_4d(g.dq), check_4d(g.dk), check_4d(g.dv);
        {
            WithoutGil nogil;
            c10::OptionalDeviceGuard device(q.device());
            check_rc(call_bwd(q, k, v, o, d_o, lse, z, scale, causal, kv_len, mask, ws, g), "flame_attn_bwd_bf16");
        }
        return triple(g);
    });
}

void call_fwd_bias(const Tensor& q, const Tensor& k, const Tensor& v, const Sizes& z, float scale, const BiasView& bias, const MaskView& mask,
                   bool want_lse, Tensor& o, Tensor& lse) {
    o = empty({z.B, z.H, z.Sq, z.D}, at::kBFloat16, q);
    if (want_lse) lse = empty({(int64_t)z.B * z.H, z.Sq}, at::kFloat, q);
    check_rc(g_api.flame_attn_fwd_bias_bf16(ptr(q), ptr(k), ptr(v), ptr(o), ptr(lse), z.B, z.H, z.Sq, z.Sk, z.D, scale, strides4(q), strides4(k),
                                            strides4(v), strides4(o), 0, 0, 0, 0, 0, bias.data, bias.dtype, bias.strides(), mask.data, mask.strides(),
                                            stream_of(q)),
             "flame_attn_fwd_bias_bf16");
}

// sdpa_with_bias(q, k, v, bias, scale | None) -> o
PyObject* py_sdpa_with_bias(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need_args(n, 5);
        const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v"), &b = tensor_arg(a[3], "bias");
        const Sizes z = sizes_of(q, k);
        check_4d(v);
        const float scale = (float)(a[4] == Py_None ? 1.0 / std::sqrt((double)z.D) : float_arg(a[4]));
        const bool as_is = b.scalar_type() == at::kFloat || b.scalar_type() == at::kBFloat16;
        const Tensor bias = as_is ? b : b.to(at::kFloat);
        const BiasView bv = bias_view(bias, z);
        Tensor o, lse;
        {
            WithoutGil nogil;
            c10::OptionalDeviceGuard device(q.device());
            const at::ScalarType orig = q.scalar_type();
            call_fwd_bias(as_bf16_view(q), as_bf16_view(k), as_bf16_view(v), z, scale, bv, MaskView(), false, o, lse);
            if (orig != at::kBFloat16) o = o.to(orig);
        }
        return THPVariable_Wrap(o);
    });
}

// attn_fwd_bias(q, k, v, scale, bias, mask, want_lse) -> (o, lse | None)
PyObject* py_attn_fwd_bias(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need_args(n, 7);
        const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v");
        const Sizes z = sizes_of(q, k);
        check_4d(v);
        const float scale = (float)float_arg(a[3]);
        const BiasView bias = bias_view(tensor_arg(a[4], "bias"), z);
        const MaskView mask = mask_view(opt_tensor_arg(a[5], "mask"), z);
        const bool want_lse = bool_arg(a[6]);
        Tensor o, lse;
        {
            WithoutGil nogil;
            c10::OptionalDeviceGuard device(q.device());
            call_fwd_bias(q, k, v, z, scale, bias, mask, want_lse, o, lse);
        }
        return pair(o, lse);
    });
}

// attn_fwd_dropout(q, k, v, scale, p, seed, causal, kv_len, mask, out, draw_chunk_q, draw_chunk_kv) -> (o, lse)
PyObject* py_attn_fwd_dropout(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need_args(n, 12);
        const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v");
        const Sizes z = sizes_of(q, k);
        check_4d(v);
        const float scale = (float)float_arg(a[3]), p = (float)float_arg(a[4]);
        const uint64_t seed = u64_arg(a[5]);
        const bool causal = bool_arg(a[6]);
        const Tensor kv_len = opt_tensor_arg(a[7], "kv_len");
        const MaskView mask = mask_view(opt_tensor_arg(a[8], "mask"), z);
        Tensor o = opt_tensor_arg(a[9], "out"), lse;
        const int cq = (int)long_arg(a[10]), ck = (int)long_arg(a[11]);
        {
            WithoutGil nogil;
            c10::OptionalDeviceGuard device(q.device());
            if (!o.defined()) o = empty({z.B, z.H, z.Sq, z.D}, at::kBFloat16, q);
            lse = empty({(int64_t)z.B * z.H, z.Sq}, at::kFloat, q);
            check_rc(g_api.flame_attn_fwd_dropout_tiled_bf16(ptr(q), ptr(k), ptr(v), ptr(o), ptr(lse), z.B, z.H, z.Sq, z.Sk, z.D, scale, strides4(q),
                                                             strides4(k), strides4(v), strides4(o), 0, 0, 0, 0, 0, causal,
                                                             static_cast<const int32_t*>(ptr(kv_len)), mask.data, mask.strides(), p, seed, cq, ck,
                                                             stream_of(q)),
                     "flame_attn_fwd_dropout_tiled_bf16");
        }
        return pair(o, lse);
    });
}

// attn_bwd_dropout(q, k, v, o, do, lse, scale, p, seed, causal, kv_len, mask, workspace, draw_chunk_q, draw_chunk_kv)
PyObject* py_attn_bwd_dropout(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need_args(n, 15);
        const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k"), &v = tensor_arg(a[2], "v"), &o = tensor_arg(a[3], "o"),
                     &d_o = tensor_arg(a[4], "do"), &lse = tensor_arg(a[5], "lse");
        const Sizes z = sizes_of(q, k);
        check_4d(v), check_4d(o), check_4d(d_o);
        const float scale = (float)float_arg(a[6]), p = (float)float_arg(a[7]);
        const uint64_t seed = u64_arg(a[8]);
        const bool causal = bool_arg(a[9]);
        const Tensor kv_len = opt_tensor_arg(a[10], "kv_len");
        const MaskView mask = mask_view(opt_tensor_arg(a[11], "mask"), z);
        Tensor ws = opt_tensor_arg(a[12], "workspace");
        const int cq = (int)long_arg(a[13]), ck = (int)long_arg(a[14]);
        Grads g;
        {
            WithoutGil nogil;
            c10::OptionalDeviceGuard device(q.device());
            if (!ws.defined()) ws = bytes_like(g_api.flame_attn_bwd_workspace_bytes(z.B, z.H, z.Sq, z.D), q);
            alloc_grads(q, z, g);
            check_rc(g_api.flame_attn_bwd_dropout_tiled_bf16(ptr(q), ptr(k), ptr(v), ptr(o), ptr(d_o), ptr(lse), ptr(g.dq), ptr(g.dk), ptr(g.dv), z.B, z.H,
                                                             z.Sq, z.Sk, z.D, scale, strides4(q), strides4(k), strides4(v), strides4(o), strides4(d_o),
                                                             strides4(g.dq), strides4(g.dk), strides4(g.dv), 0, 0, 0, 0, 0, 0, 0, 0, 0, causal,
                                                             static_cast<const int32_t*>(ptr(kv_len)), mask.data, mask.strides(), p, seed, cq, ck, ptr(ws),
                                                             (size_t)ws.numel(), stream_of(q)),
                     "flame_attn_bwd_dropout_tiled_bf16");
        }
        return triple(g);
    });
}

// sage_quant(q, k, smooth_k, want_ks, row_elems) -> dict
PyObject* py_sage_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need_args(n, 5);
        const Tensor &q = tensor_arg(a[0], "q"), &k = tensor_arg(a[1], "k");
        const Sizes z = sizes_of(q, k);
        const bool smooth = bool_arg(a[2]), want_ks = bool_arg(a[3]);
        const int64_t Dp = long_arg(a[4]);
        Tensor qi, ki, sq, sk, km, ks;
        {
            WithoutGil nogil;
            c10::OptionalDeviceGuard device(q.device());
            auto cut = [&](Tensor t) { return t.narrow(-1, 0, std::min<int64_t>(z.D, Dp)); };      // the columns of the real head dim
            qi = cut(empty({z.B, z.H, z.Sq, Dp}, at::kChar, q));
            ki = cut(empty({z.B, z.H, z.Sk, Dp}, at::kChar, q));
            sq = empty({z.B, z.H, (z.Sq + 127) / 128}, at::kFloat, q);
            sk = empty({z.B, z.H, (z.Sk + 63) / 64}, at::kFloat, q);
            km = cut(empty({z.B, z.H, Dp}, at::kFloat, q));
            if (want_ks) ks = cut(empty({z.B, z.H, z.Sk, Dp}, at::kBFloat16, q));
            check_rc(g_api.flame_sage_quant_qk_int8_ks(ptr(q), ptr(k), z.B, z.H, z.Sq, z.Sk, z.D, strides4(q), strides4(k), 0, 0, smooth, ptr(qi), ptr(ki),
                                                       ptr(sq), ptr(sk), ptr(km), ptr(ks), stream_of(q)),
                     "flame_sage_quant_qk_int8_ks");
        }
        PyObject* d = PyDict_New();
        auto put = [&](const char* name, const Tensor& t) {
            PyObject* o = THPVariable_Wrap(t);
            PyDict_SetItemString(d, name, o);
            Py_DECREF(o);
        };
        put("qi8", qi), put("ki8", ki), put("sq", sq), put("sk", sk), put("kmean", km);
        if (want_ks) put("ks", ks);
        return d;
    });
}

// sage_fwd(qi8, ki8, sq, sk, v, scale, causal, kv_len, want_lse, out, bias) -> (o, lse | None)
PyObject* py_sage_fwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need_args(n, 11);
        const Tensor &qi = tensor_arg(a[0], "qi8"), &ki = tensor_arg(a[1], "ki8"), &sq = tensor_arg(a[2], "sq"), &sk = tensor_arg(a[3], "sk"),
                     &v = tensor_arg(a[4], "v");
        const Sizes z = sizes_of(qi, ki);
        check_4d(v);
        const float scale = (float)float_arg(a[5]);
        const bool causal = bool_arg(a[6]);
        const Tensor kv_len = opt_tensor_arg(a[7], "kv_len");
        const bool want_lse = bool_arg(a[8]);
        Tensor o = opt_tensor_arg(a[9], "out"), lse;
        const BiasView bias = bias_view(opt_tensor_arg(a[10], "bias"), z);
        {
            WithoutGil nogil;
            c10::OptionalDeviceGuard device(v.device());
            if (!o.defined()) o = empty({z.B, z.H, z.Sq, z.D}, at::kBFloat16, v);
            if (want_lse) lse = empty({(int64_t)z.B * z.H, z.Sq}, at::kFloat, v);
            check_rc(g_api.flame_sage_attn_fwd_bias_int8(ptr(qi), ptr(ki), ptr(sq), ptr(sk), ptr(v), ptr(o), ptr(lse), z.B, z.H, z.Sq, z.Sk, z.D, scale,
                                                         strides4(v), strides4(o), 0, 0, causal, static_cast<const int32_t*>(ptr(kv_len)), bias.data,
                                                         bias.dtype, bias.strides(), stream_of(v)),
                     "flame_sage_attn_fwd_bias_int8");
        }
        return pair(o, lse);
    });
}

// prep_rmsnorm_rope(x_bnhd, weight, cos, sin, eps, apply_norm, out) -> [B,H,N,D]
PyObject* py_prep(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need_args(n, 7);
        const Tensor& x = tensor_arg(a[0], "x_bnhd");
        check_4d(x);
        const Tensor w = opt_tensor_arg(a[1], "weight"), cos = opt_tensor_arg(a[2], "cos"), sin = opt_tensor_arg(a[3], "sin");
        const float eps = (float)float_arg(a[4]);
        const bool norm = bool_arg(a[5]);
        Tensor out = opt_tensor_arg(a[6], "out");
        const int64_t B = x.size(0), N = x.size(1), H = x.size(2), D = x.size(3);
        int tdt = FLAME_ATTN_DTYPE_BF16;
        if (cos.defined()) {
            if (!sin.defined() || cos.scalar_type() != sin.scalar_type() || cos.dim() != 2 || cos.sizes() != sin.sizes() || cos.size(0) != N ||
                cos.size(1) != D / 2)
                fail(PyExc_ValueError, "cos/sin must both be [N, D/2] of one dtype");
            if (!cos.is_contiguous() || !sin.is_contiguous()) fail(PyExc_ValueError, "cos/sin must be contiguous");
            if (cos.scalar_type() == at::kFloat) tdt = FLAME_ATTN_DTYPE_F32;
        }
        if (out.defined()) check_4d(out);
        {
            WithoutGil nogil;
            c10::OptionalDeviceGuard device(x.device());
            if (!out.defined()) out = empty({B, H, N, D}, at::kBFloat16, x);
            const int64_t xs[4] = {x.stride(0), x.stride(2), x.stride(1), x.stride(3)};      // the same memory seen as [B,H,N,D]
            check_rc(g_api.flame_attn_prep_rmsnorm_rope_bf16(ptr(x), ptr(w), ptr(cos), cos.defined() ? ptr(sin) : nullptr, tdt, ptr(out), (int)B, (int)H,
                                                             (int)N, (int)D, eps, norm, xs, strides4(out), 0, 0, stream_of(x)),
                     "flame_attn_prep_rmsnorm_rope_bf16");
        }
        return THPVariable_Wrap(out);
    });
}

// fp8(x, scale, out, encode) -> codes or values
PyObject* py_fp8(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need_args(n, 4);
        const Tensor& x = tensor_arg(a[0], "x");
        const float scale = (float)float_arg(a[1]);
        Tensor out = opt_tensor_arg(a[2], "out");
        const bool encode = bool_arg(a[3]);
        const at::ScalarType from = encode ? at::kBFloat16 : at::kByte, to = encode ? at::kByte : at::kBFloat16;
        check_that(x.scalar_type() == from && x.is_contiguous(), "a contiguous tensor of the source type is expected");
        check_that(!out.defined() || (out.scalar_type() == to && out.is_contiguous() && out.numel() == x.numel()),
                   "out is a contiguous tensor of the result type with as many elements");
        {
            WithoutGil nogil;
            c10::OptionalDeviceGuard device(x.device());
            if (!out.defined()) out = empty(x.sizes(), to, x);
            const size_t count = (size_t)x.numel();
            if (encode) check_rc(g_api.flame_bf16_to_fp8(ptr(x), ptr(out), scale, count, stream_of(x)), "flame_bf16_to_fp8");
            else check_rc(g_api.flame_fp8_to_bf16(ptr(x), ptr(out), scale, count, stream_of(x)), "flame_fp8_to_bf16");
        }
        return THPVariable_Wrap(out);
    });
}

// bind(dlopen handle of the library, the exception class)
PyObject* py_bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        need_args(n, 2);
        void* lib = PyLong_AsVoidPtr(a[0]);
        if (!lib && PyErr_Occurred()) throw PyErrorSet{};
        const char* missing = nullptr;
#define FLAME_HOST_LOOK_UP(name)                                              \
    g_api.name = reinterpret_cast<decltype(g_api.name)>(dlsym(lib, #name));   \
    if (!g_api.name) missing = #name;
        FLAME_HOST_ENTRY_POINTS(FLAME_HOST_LOOK_UP)
#undef FLAME_HOST_LOOK_UP
        if (missing) {
            PyErr_Format(PyExc_RuntimeError, "the attention library does not export %s", missing);
            throw PyErrorSet{};
        }
        Py_XINCREF(a[1]);
        Py_XDECREF(g_error_class);
        g_error_class = a[1];
        return Py_NewRef(Py_None);
    });
}

#define FLAME_HOST_METHOD(name, f) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {FLAME_HOST_METHOD("bind", py_bind),
                           FLAME_HOST_METHOD("sdpa", py_sdpa),
                           FLAME_HOST_METHOD("sdpa_with_bias", py_sdpa_with_bias),
                           FLAME_HOST_METHOD("attn_fwd", py_attn_fwd),
                           FLAME_HOST_METHOD("attn_bwd", py_attn_bwd),
                           FLAME_HOST_METHOD("attn_fwd_bias", py_attn_fwd_bias),
                           FLAME_HOST_METHOD("attn_fwd_dropout", py_attn_fwd_dropout),
                           FLAME_HOST_METHOD("attn_bwd_dropout", py_attn_bwd_dropout),
                           FLAME_HOST_METHOD("sage_quant", py_sage_quant),
                           FLAME_HOST_METHOD("sage_fwd", py_sage_fwd),
                           FLAME_HOST_METHOD("prep_rmsnorm_rope", py_prep),
                           FLAME_HOST_METHOD("fp8", py_fp8),
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_flame_torch_host", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__flame_torch_host() { return PyModule_Create(&g_module); }
