// Host layer of tyr_amd.gpu in native code: argument checks, output and scratch allocation and the call of the C ABI
// (include/tyr_hip.h) for torch tensors, as one CPython extension module `_tyr_torch`.
//
// What bounds it: host time per call.  A kernel launch costs 2.4 us on this host by itself; the same steps written in
// Python (attribute reads, torch.empty, current_stream, ctypes conversion) brought a call to 8.5 (copy) .. 20 us
// (attention backward), longer than many of the kernels they launch.  Here arguments arrive by METH_FASTCALL, tensors are
// read through their TensorImpl, and outputs come straight from the caching allocator's factory without a dispatcher walk.
//
// The checks and their messages are those of the reference's generated launcher (Tyr/GPU/Codegen/Attribute.lean:334-336:
// device, contiguity, rank <= 4), in the same order for every argument.  Scratch is a caching-allocator block of the
// current stream, dropped on return: work queued later on that stream is ordered behind the kernels that use it.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <atomic>
#include <cmath>
#include <string>

#include "../../include/tyr_hip.h"
#include "torch_scratch.hpp"

namespace {

struct Failure {                      // becomes TyrGpuError
    std::string what;
};
[[noreturn]] void fail(std::string what) { throw Failure{std::move(what)}; }

// The C ABI.  It is not linked in: the library can be another build, and is opened by the first call of one of its
// functions, not by the import of the package.  A build without some of them serves the calls that need only the others.
std::string g_library;                // path, from load()
PyObject* g_error = nullptr;          // tyr_amd.gpu.TyrGpuError

void* library() {
    static void* const handle = [] {  // a failed attempt throws and is repeated by the next call
        void* h = dlopen(g_library.c_str(), RTLD_NOW | RTLD_LOCAL);
        if (!h) fail(std::string(dlerror()) + " (build it with `make -C tyr_amd/csrc`; tyr_amd has no CPU or PyTorch fallback)");
        return h;
    }();
    return handle;
}
template <class F> class Symbol;
template <class R, class... A> class Symbol<R (*)(A...)> {
    const char* name_;
    mutable std::atomic<R (*)(A...)> f_{nullptr};
public:
    explicit Symbol(const char* name) : name_(name) {}
    R operator()(A... a) const {
        R (*f)(A...) = f_.load(std::memory_order_relaxed);
        if (!f) {
            f = reinterpret_cast<R (*)(A...)>(dlsym(library(), name_));
            if (!f) fail(g_library + " does not export " + name_);
            f_.store(f, std::memory_order_relaxed);
        }
        return f(a...);
    }
};
#define TYR_ENTRY_POINTS(X)                                                                                                  \
    X(tyr_hip_strerror) X(tyr_hip_flash_attn_fwd_gqa) X(tyr_hip_flash_attn_fwd_mask) X(tyr_hip_flash_attn_bwd_full_workspace_bytes) \
    X(tyr_hip_flash_attn_bwd_parts_workspace_bytes) X(tyr_hip_flash_attn_bwd_workspace_bytes)                                \
    X(tyr_hip_flash_attn_bwd_gqa) X(tyr_hip_flash_attn_bwd_mask) X(tyr_hip_gqa_decode_workspace_bytes)                        \
    X(tyr_hip_gqa_decode_varlen) X(tyr_hip_decode_rope_append) X(tyr_hip_rope_fwd) X(tyr_hip_layernorm_residual)             \
    X(tyr_hip_copy) X(tyr_hip_gemm_workspace_bytes) X(tyr_hip_gemm_bf16_batched_ws) X(tyr_hip_gemm_fp8_ws)                    \
    X(tyr_hip_mse_loss_grad_workspace_bytes) X(tyr_hip_mse_loss_grad) X(tyr_hip_sgd_step)
const struct Api {
#define X(f) Symbol<decltype(&::f)> f{#f};
    TYR_ENTRY_POINTS(X)
#undef X
} api;

void check_status(int rc, const char* what) {
    if (rc != 0)
        fail(std::string(what) + ": " + api.tyr_hip_strerror(rc) + " (status " + std::to_string(rc) + ")");
}

struct NoGil {                        // ctypes calls ran without the GIL: keep launches of several threads concurrent
    PyThreadState* s = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(s); }
};

const at::Tensor& tensor(PyObject* o, const char* name) {
    if (!THPVariable_Check(o)) fail(std::string(name) + " must be a tensor");
    return THPVariable_Unpack(o);
}

void check(const at::Tensor& t, const char* name, at::ScalarType dtype, int ndim = -1) {
    if (!t.is_cuda()) fail(std::string(name) + " must be a CUDA tensor");
    if (!t.is_contiguous()) fail(std::string(name) + " must be contiguous");
    if (t.dim() > 4) fail(std::string(name) + " must have dim <= 4");
    if (ndim >= 0 && t.dim() != ndim) fail(std::string(name) + " must have dim == " + std::to_string(ndim));
    if (t.scalar_type() != dtype) fail(std::string(name) + " must have dtype torch." + torch::getTHPDtype(dtype)->name);
}
const at::Tensor& checked(PyObject* o, const char* name, at::ScalarType dtype, int ndim = -1) {
    const at::Tensor& t = tensor(o, name);
    check(t, name, dtype, ndim);
    return t;
}

at::Tensor empty(at::IntArrayRef sizes, at::ScalarType dtype, const at::Tensor& like) {
    return at::Tensor(at::detail::empty_cuda(sizes, dtype, like.device(), std::nullopt));
}
at::Tensor empty_like(const at::Tensor& t) { return empty(t.sizes(), t.scalar_type(), t); }
at::Tensor scratch(size_t bytes, const at::Tensor& like) { return empty({(int64_t)std::max<size_t>(bytes, 16)}, at::kByte, like); }

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

bool truth(PyObject* o) {
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw python_error();
    return v != 0;
}
int64_t integer(PyObject* o) {
    PyObject* i = PyNumber_Long(o);
    if (!i) throw python_error();
    const int64_t v = (int64_t)PyLong_AsUnsignedLongLongMask(i);
    Py_DECREF(i);
    if (PyErr_Occurred()) throw python_error();
    return v;
}
double real(PyObject* o) {
    if (PyFloat_CheckExact(o)) return PyFloat_AS_DOUBLE(o);
    PyObject* f = PyNumber_Float(o);
    if (!f) throw python_error();
    const double v = PyFloat_AS_DOUBLE(f);
    Py_DECREF(f);
    return v;
}
float attn_scale(PyObject* o, int64_t D) { return (float)(o == Py_None ? 1.0 / std::sqrt((double)D) : real(o)); }

PyObject* wrap(at::Tensor t) { return THPVariable_Wrap(std::move(t)); }
template <class... T>
PyObject* wrap_tuple(T&&... t) {
    PyObject* items[] = {wrap(std::forward<T>(t))...};
    PyObject* out = PyTuple_New(sizeof...(T));
    for (size_t i = 0; i < sizeof...(T); ++i) PyTuple_SET_ITEM(out, i, items[i]);
    return out;
}

// ---- attention
const int32_t* lengths(PyObject* o, int64_t B) {
    if (o == Py_None) return nullptr;
    const at::Tensor& t = checked(o, "kvLens", at::kInt, 1);
    if (t.numel() != B) fail("kvLens must hold one length per sequence");
    return static_cast<const int32_t*>(t.data_ptr());
}
// [B, N] key mask (bool or uint8, nonzero = visible)
const uint8_t* mask_bytes(PyObject* o, int64_t B, int64_t N, int64_t window, bool has_lens) {
    if (window || has_lens) fail("a key mask cannot be combined with a window or key lengths");
    const at::Tensor& t = tensor(o, "keyMask");
    if (t.scalar_type() != at::kBool && t.scalar_type() != at::kByte) fail("keyMask must have dtype torch.bool or torch.uint8");
    check(t, "keyMask", t.scalar_type(), 2);
    if (t.size(0) != B || t.size(1) != N) fail("keyMask must have shape [B, N]");
    return static_cast<const uint8_t*>(t.data_ptr());
}

// (q, k, v, causal, scale, window, kv_lens, key_mask)
PyObject* flash_attn_fwd(PyObject* const* a) {
    const at::Tensor &q = checked(a[0], "q", at::kBFloat16, 4), &k = checked(a[1], "k", at::kBFloat16, 4),
                     &v = checked(a[2], "v", at::kBFloat16, 4);
    const int64_t B = q.size(0), Hq = q.size(1), N = q.size(2), D = q.size(3), Hkv = k.size(1);
    if (k.sizes() != v.sizes() || k.size(0) != B || k.size(2) != N || k.size(3) != D)
        fail("k, v must have shape [B, Hkv, N, D] matching q's B, N, D");
    if (Hkv == 0 || Hq % Hkv != 0) fail("the number of query heads must be a multiple of the number of kv heads");
    const bool causal = truth(a[3]);
    const float scale = attn_scale(a[4], D);
    const int64_t window = integer(a[5]);
    const int32_t* lens = lengths(a[6], B);
    const uint8_t* mask = a[7] == Py_None ? nullptr : mask_bytes(a[7], B, N, window, lens != nullptr);
    at::Tensor o, lse;
    int rc;
    {
        NoGil nogil;
        o = empty_like(q);
        lse = empty({B, Hq, N}, at::kFloat, q);
        rc = mask ? api.tyr_hip_flash_attn_fwd_mask(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), (float*)lse.data_ptr(), B, Hq,
                                                    Hkv, N, D, causal, mask, scale, stream())
                  : api.tyr_hip_flash_attn_fwd_gqa(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), (float*)lse.data_ptr(), B, Hq,
                                                   Hkv, N, D, causal, window, lens, scale, stream());
    }
    check_status(rc, "flashAttnFwd");
    return wrap_tuple(std::move(o), std::move(lse));
}

// (q, k, v, o, lse, d_o, causal, scale, window, kv_lens, key_mask)
PyObject* flash_attn_bwd(PyObject* const* a) {
    const at::Tensor &q = checked(a[0], "q", at::kBFloat16, 4), &k = checked(a[1], "k", at::kBFloat16, 4),
                     &v = checked(a[2], "v", at::kBFloat16, 4), &o = checked(a[3], "o", at::kBFloat16, 4),
                     &d_o = checked(a[5], "dO", at::kBFloat16, 4);
    if (o.sizes() != q.sizes() || d_o.sizes() != q.sizes() || k.sizes() != v.sizes())
        fail("q, o, dO must have the same shape [B, Hq, N, D] and k, v the same shape [B, Hkv, N, D]");
    const at::Tensor& lse = checked(a[4], "lse", at::kFloat, 3);
    const int64_t B = q.size(0), Hq = q.size(1), N = q.size(2), D = q.size(3), Hkv = k.size(1);
    if (k.size(0) != B || k.size(2) != N || k.size(3) != D)
        fail("q, k, v, o, dO must have the same shape [B, H, N, D] (k, v may have fewer heads)");
    if (Hkv == 0 || Hq % Hkv != 0) fail("the number of query heads must be a multiple of the number of kv heads");
    if (lse.size(0) != B || lse.size(1) != Hq || lse.size(2) != N) fail("lse must have shape [B, H, N]");
    const bool causal = truth(a[6]);
    const float scale = attn_scale(a[7], D);
    const int64_t window = integer(a[8]);
    const int32_t* lens = lengths(a[9], B);
    const uint8_t* mask = a[10] == Py_None ? nullptr : mask_bytes(a[10], B, N, window, lens != nullptr);
    at::Tensor dq, dk, dv;
    int rc;
    {
        NoGil nogil;
        dq = empty_like(q);
        dk = empty_like(k);
        dv = empty_like(k);
        const at::Tensor ws = tyr_torch::take_largest(api.tyr_hip_flash_attn_bwd_full_workspace_bytes(B, Hq, Hkv, N, D, causal, window),
                                                      api.tyr_hip_flash_attn_bwd_parts_workspace_bytes(B, Hq, Hkv, N, D, causal, window),
                                                      api.tyr_hip_flash_attn_bwd_workspace_bytes(B, Hq, N, D), q.device().index(),
                                                      [&](size_t bytes) { return scratch(bytes, q); });
        const float* lse_p = static_cast<const float*>(lse.data_ptr());
        rc = mask ? api.tyr_hip_flash_attn_bwd_mask(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), d_o.data_ptr(), lse_p,
                                                    dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), B, Hq, Hkv, N, D, causal, mask, scale,
                                                    ws.data_ptr(), ws.numel(), stream())
                  : api.tyr_hip_flash_attn_bwd_gqa(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), d_o.data_ptr(), lse_p,
                                                   dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), B, Hq, Hkv, N, D, causal, window, lens, scale,
                                                   ws.data_ptr(), ws.numel(), stream());
    }
    check_status(rc, "flashAttnBwd");
    return wrap_tuple(std::move(dq), std::move(dk), std::move(dv));
}

// (q, k, v, scale, num_splits, kv_len, kv_lens, window)
PyObject* gqa_decode(PyObject* const* a) {
    const at::Tensor &q = checked(a[0], "q", at::kBFloat16, 4), &k = checked(a[1], "k", at::kBFloat16, 4),
                     &v = checked(a[2], "v", at::kBFloat16, 4);
    const int64_t B = q.size(0), Hq = q.size(1), D = q.size(3);
    if (q.size(2) != 1) fail("q must have shape [B, Hq, 1, D]");
    if (k.sizes() != v.sizes() || k.size(0) != B || k.size(3) != D) fail("k, v must have shape [B, Hkv, L, D]");
    const int64_t Hkv = k.size(1), Lmax = k.size(2);
    const float scale = attn_scale(a[3], D);
    const int64_t splits = integer(a[4]);
    const int64_t L = a[5] == Py_None ? Lmax : integer(a[5]);
    const int32_t* lens = lengths(a[6], B);
    const int64_t window = integer(a[7]);
    at::Tensor o, lse;
    int rc;
    {
        NoGil nogil;
        o = empty_like(q);
        lse = empty({B, Hq}, at::kFloat, q);
        const at::Tensor ws =
            scratch(api.tyr_hip_gqa_decode_workspace_bytes(B, Hq, std::max<int64_t>(Hkv, 1), std::max<int64_t>(L, 1), D, splits), q);
        rc = api.tyr_hip_gqa_decode_varlen(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), (float*)lse.data_ptr(), B, Hq, Hkv, L, D,
                                           Lmax, lens, window, scale, splits, ws.data_ptr(), ws.numel(), stream());
    }
    check_status(rc, "gqaDecode");
    return wrap_tuple(std::move(o), std::move(lse));
}

// (q, k_new, v_new, cos, sin, k_cache, v_cache, pos)
PyObject* decode_rope_append(PyObject* const* a) {
    const at::Tensor &q = checked(a[0], "q", at::kBFloat16, 4), &kn = checked(a[1], "kNew", at::kBFloat16, 4),
                     &vn = checked(a[2], "vNew", at::kBFloat16, 4), &kc = checked(a[5], "kCache", at::kBFloat16, 4),
                     &vc = checked(a[6], "vCache", at::kBFloat16, 4);
    const at::Tensor &cos = checked(a[3], "cos", at::kFloat), &sin = checked(a[4], "sin", at::kFloat);
    const int64_t B = kc.size(0), Hkv = kc.size(1), Lmax = kc.size(2), D = kc.size(3);
    if (vc.sizes() != kc.sizes()) fail("k and v caches must have the same shape");
    if (q.size(0) != B || q.size(3) != D || (q.size(1) != 1 && q.size(2) != 1)) fail("q must be [B, Hq, 1, D] or [B, 1, Hq, D]");
    const int64_t Hq = q.size(1) * q.size(2);
    for (const at::Tensor* t : {&kn, &vn})
        if (t->numel() != B * Hkv * D || t->size(3) != D) fail("kNew and vNew must hold B*Hkv rows of D elements");
    if (cos.numel() != D / 2 || sin.numel() != D / 2) fail("cos and sin must hold D/2 elements (the table row of this position)");
    const int64_t pos = integer(a[7]);
    if (pos < 0 || pos >= Lmax) fail("pos is outside the cache");
    at::Tensor q_out;
    int rc;
    {
        NoGil nogil;
        q_out = empty_like(q);
        rc = api.tyr_hip_decode_rope_append(q.data_ptr(), kn.data_ptr(), vn.data_ptr(), (const float*)cos.data_ptr(),
                                            (const float*)sin.data_ptr(), q_out.data_ptr(), kc.data_ptr(), vc.data_ptr(), B, Hq, Hkv, D,
                                            Lmax, pos, stream());
    }
    check_status(rc, "decodeRopeAppend");
    return wrap(std::move(q_out));
}

// ---- row kernels
// (x, cos, sin)
PyObject* rope_fwd(PyObject* const* a) {
    const at::Tensor& x = tensor(a[0], "x");
    if (x.scalar_type() != at::kFloat && x.scalar_type() != at::kBFloat16) fail("x must have dtype float32 or bfloat16");
    check(x, "x", x.scalar_type(), 4);
    const at::Tensor &cos = checked(a[1], "cos", at::kFloat, 2), &sin = checked(a[2], "sin", at::kFloat, 2);
    const int64_t B = x.size(0), S = x.size(1), H = x.size(2), D = x.size(3);
    for (const at::Tensor* t : {&cos, &sin})
        if (t->size(0) != S || t->size(1) != D / 2) fail("cos and sin must have shape [S, D/2]");
    at::Tensor y;
    int rc;
    {
        NoGil nogil;
        y = empty_like(x);
        rc = api.tyr_hip_rope_fwd(x.data_ptr(), (const float*)cos.data_ptr(), (const float*)sin.data_ptr(), y.data_ptr(), B, S, H, D,
                                  x.scalar_type() == at::kBFloat16 ? TYR_HIP_BF16 : TYR_HIP_F32, stream());
    }
    check_status(rc, "applyRotaryEmb");
    return wrap(std::move(y));
}

// (x, residual, weight, bias, eps)
PyObject* layernorm_residual(PyObject* const* a) {
    const at::Tensor &x = checked(a[0], "x", at::kBFloat16), &res = checked(a[1], "residual", at::kBFloat16),
                     &w = checked(a[2], "weight", at::kBFloat16), &b = checked(a[3], "bias", at::kBFloat16);
    const float eps = (float)real(a[4]);
    if (x.dim() == 0) fail("x must have dim >= 1");
    const int64_t d = x.size(-1);
    if (res.sizes() != x.sizes() || w.dim() != 1 || w.size(0) != d || b.dim() != 1 || b.size(0) != d)
        fail("residual must match x, weight and bias must be [d_model]");
    at::Tensor out, out_resid;
    int rc;
    {
        NoGil nogil;
        out = empty_like(x);
        out_resid = empty_like(x);
        rc = api.tyr_hip_layernorm_residual(x.data_ptr(), res.data_ptr(), w.data_ptr(), b.data_ptr(), out.data_ptr(), out_resid.data_ptr(),
                                            d ? x.numel() / d : 0, d, eps, stream());
    }
    check_status(rc, "fusedLayerNormResidual");
    return wrap_tuple(std::move(out), std::move(out_resid));
}

// (src)
PyObject* copy(PyObject* const* a) {
    const at::Tensor& src = tensor(a[0], "input");
    check(src, "input", src.scalar_type());
    at::Tensor dst;
    int rc;
    {
        NoGil nogil;
        dst = empty_like(src);
        rc = api.tyr_hip_copy(src.data_ptr(), dst.data_ptr(), src.numel() * src.element_size(), stream());
    }
    check_status(rc, "copy");
    return wrap(std::move(dst));
}

// ---- products
// B is [..., K, N], or [..., N, K] when transposed
struct Extents { int64_t M, N, K; };
Extents extents(const at::Tensor& a, const at::Tensor& b, bool trans_b) {
    const int64_t M = a.size(-2), K = a.size(-1), N = trans_b ? b.size(-2) : b.size(-1), Kb = trans_b ? b.size(-1) : b.size(-2);
    if (Kb != K) fail("a and b have mismatched inner dimensions");
    return {M, N, K};
}

// scratch for split-K partials, where the library splits this product
struct Partials {
    size_t bytes;
    at::Tensor block;
    Partials(int64_t batch, const Extents& e, int elem_bytes, bool trans_b, const at::Tensor& like)
        : bytes(api.tyr_hip_gemm_workspace_bytes(batch, e.M, e.N, e.K, elem_bytes, trans_b)) {
        if (bytes) block = scratch(bytes, like);
    }
    void* ptr() const { return bytes ? block.data_ptr() : TYR_HIP_ANY_ORDER; }
};

// (a, b, trans_b)
PyObject* gemm_bf16(PyObject* const* a) {
    const at::Tensor &x = checked(a[0], "a", at::kBFloat16, 2), &y = checked(a[1], "b", at::kBFloat16, 2);
    const bool trans_b = truth(a[2]);
    const Extents e = extents(x, y, trans_b);
    at::Tensor c;
    int rc;
    {
        NoGil nogil;
        c = empty({e.M, e.N}, at::kBFloat16, x);
        const Partials ws(1, e, 2, trans_b, x);
        rc = api.tyr_hip_gemm_bf16_batched_ws(x.data_ptr(), y.data_ptr(), c.data_ptr(), 1, e.M, e.N, e.K, 0, 0, 0, trans_b, ws.ptr(),
                                              ws.bytes, stream());
    }
    check_status(rc, "gemmBf16");
    return wrap(std::move(c));
}

// (a, b, trans_b)
PyObject* matmul_bf16(PyObject* const* a) {
    const at::Tensor &x = checked(a[0], "a", at::kBFloat16), &y = checked(a[1], "b", at::kBFloat16);
    if (x.dim() < 2 || y.dim() < 2) fail("a and b must have dim >= 2");
    if (x.dim() == 2 && y.dim() == 2) return gemm_bf16(a);
    if (y.dim() != 2 && (y.dim() != x.dim() || y.sizes().slice(0, y.dim() - 2) != x.sizes().slice(0, x.dim() - 2)))
        fail("b must be a matrix or share a's leading extents");
    if (x.dim() == 2) fail("a must carry the batch extents");
    const bool trans_b = truth(a[2]);
    const Extents e = extents(x, y, trans_b);
    const int64_t batch = e.M * e.K != 0 ? x.numel() / (e.M * e.K) : 0;
    at::DimVector sizes(x.sizes().begin(), x.sizes().end());
    sizes.back() = e.N;
    at::Tensor c;
    int rc;
    {
        NoGil nogil;
        c = empty(sizes, at::kBFloat16, x);
        const Partials ws(batch, e, 2, trans_b, x);
        rc = api.tyr_hip_gemm_bf16_batched_ws(x.data_ptr(), y.data_ptr(), c.data_ptr(), batch, e.M, e.N, e.K, e.M * e.K,
                                              y.dim() == 2 ? 0 : e.K * e.N, e.M * e.N, trans_b, ws.ptr(), ws.bytes, stream());
    }
    check_status(rc, "matmul");
    return wrap(std::move(c));
}

PyObject* fp8(PyObject* pa, PyObject* pb, float scale, PyObject* row, PyObject* col, at::ScalarType out, bool trans_b, const char* what) {
    const at::Tensor &x = checked(pa, "a", at::kFloat8_e4m3fn, 2), &y = checked(pb, "b", at::kFloat8_e4m3fn, 2);
    const Extents e = extents(x, y, trans_b);
    int kind = TYR_HIP_OUT_BF16;
    if (out == at::kFloat) kind = TYR_HIP_OUT_F32;
    else if (out == at::kFloat8_e4m3fn) kind = TYR_HIP_OUT_E4M3;
    else if (out != at::kBFloat16) fail("out_dtype must be bfloat16, float32 or float8_e4m3fn");
    const float *rs = nullptr, *cs = nullptr;
    if (row != Py_None) {
        const at::Tensor& t = checked(row, "rowScale", at::kFloat, 1);
        if (t.numel() != e.M) fail("rowScale must hold one scale per row");
        rs = static_cast<const float*>(t.data_ptr());
    }
    if (col != Py_None) {
        const at::Tensor& t = checked(col, "colScale", at::kFloat, 1);
        if (t.numel() != e.N) fail("colScale must hold one scale per column");
        cs = static_cast<const float*>(t.data_ptr());
    }
    at::Tensor c;
    int rc;
    {
        NoGil nogil;
        c = empty({e.M, e.N}, out, x);
        const Partials ws(1, e, 1, trans_b, x);
        rc = api.tyr_hip_gemm_fp8_ws(x.data_ptr(), y.data_ptr(), c.data_ptr(), e.M, e.N, e.K, scale, rs, cs, kind, trans_b, ws.ptr(),
                                     ws.bytes, stream());
    }
    check_status(rc, what);
    return wrap(std::move(c));
}
// (aq, bq, scale_a, scale_b, trans_b)
PyObject* gemm_fp8(PyObject* const* a) {
    return fp8(a[0], a[1], (float)real(a[2]) * (float)real(a[3]), Py_None, Py_None, at::kBFloat16, truth(a[4]), "gemmFp8");
}
// (aq, bq, row_scale, col_scale, scale, out_dtype, trans_b)
PyObject* gemm_fp8_scaled(PyObject* const* a) {
    if (!THPDtype_Check(a[5])) fail("out_dtype must be bfloat16, float32 or float8_e4m3fn");
    return fp8(a[0], a[1], (float)real(a[4]), a[2], a[3], reinterpret_cast<THPDtype*>(a[5])->scalar_type, truth(a[6]), "gemmFp8Scaled");
}

// ---- train step
// (out, target)
PyObject* mse_loss_grad(PyObject* const* a) {
    const at::Tensor &o = checked(a[0], "out", at::kBFloat16), &t = checked(a[1], "target", at::kBFloat16);
    if (o.sizes() != t.sizes()) fail("out and target must have the same shape");
    at::Tensor d_o, loss;
    int rc;
    {
        NoGil nogil;
        d_o = empty_like(o);
        loss = empty({}, at::kFloat, o);
        const at::Tensor ws = scratch(api.tyr_hip_mse_loss_grad_workspace_bytes(o.numel()), o);
        rc = api.tyr_hip_mse_loss_grad(o.data_ptr(), t.data_ptr(), d_o.data_ptr(), (float*)loss.data_ptr(), o.numel(), ws.data_ptr(),
                                       ws.numel(), stream());
    }
    check_status(rc, "lossAndGradOut");
    return wrap_tuple(std::move(loss), std::move(d_o));
}
// (param, grad, lr, in_place)
PyObject* sgd_step(PyObject* const* a) {
    const at::Tensor &p = checked(a[0], "param", at::kFloat), &g = checked(a[1], "grad", at::kBFloat16);
    if (p.sizes() != g.sizes()) fail("param and grad must have the same shape");
    const float lr = (float)real(a[2]);
    const bool in_place = truth(a[3]);
    at::Tensor out, low;
    int rc;
    {
        NoGil nogil;
        out = in_place ? p : empty_like(p);
        low = empty_like(g);
        rc = api.tyr_hip_sgd_step((const float*)p.data_ptr(), g.data_ptr(), lr, (float*)out.data_ptr(), low.data_ptr(), p.numel(), stream());
    }
    check_status(rc, "sgdUpdate");
    return wrap_tuple(std::move(out), std::move(low));
}

// ---- module
template <PyObject* (*F)(PyObject* const*), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != N) {
        PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", N, n);
        return nullptr;
    }
    HANDLE_TH_ERRORS
    try {
        return F(args);
    } catch (const Failure& e) {
        PyErr_SetString(g_error, e.what.c_str());
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}

// load(path of libtyr_hip.so, exception class): remembers both
PyObject* load(PyObject*, PyObject* args) {
    const char* path = nullptr;
    PyObject* error = nullptr;
    if (!PyArg_ParseTuple(args, "sO", &path, &error)) return nullptr;
    g_library = path;
    Py_INCREF(error);
    Py_XDECREF(g_error);
    g_error = error;
    Py_RETURN_NONE;
}

#define TYR_METHOD(f, n) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&entry<f, n>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"load", load, METH_VARARGS, nullptr},
    TYR_METHOD(flash_attn_fwd, 8), TYR_METHOD(flash_attn_bwd, 11), TYR_METHOD(gqa_decode, 8), TYR_METHOD(decode_rope_append, 8),
    TYR_METHOD(rope_fwd, 3), TYR_METHOD(layernorm_residual, 5), TYR_METHOD(copy, 1), TYR_METHOD(gemm_bf16, 3),
    TYR_METHOD(matmul_bf16, 3), TYR_METHOD(gemm_fp8, 5), TYR_METHOD(gemm_fp8_scaled, 7), TYR_METHOD(mse_loss_grad, 2),
    TYR_METHOD(sgd_step, 4), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_tyr_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__tyr_torch() { return PyModule_Create(&module); }
