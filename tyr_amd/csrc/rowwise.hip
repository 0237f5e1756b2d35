// Memory-bound row kernels around the attention path (gfx950): device copy, rotary embedding,
// fused residual + LayerNorm, and the decode step's "rotate q and k, append k and v to the cache".
//
// Reference semantics restated here:
//   copy           Tyr/GPU/Kernels/Copy.lean:16-27 (copy64x64: out = in, one f32 tile per block)
//   rotary         cc/src/tyr.cpp:3837-3873 (lean_torch_apply_rotary_emb): x = [x1 | x2] split in
//                  halves along head_dim, y1 = x1 cos - x2 sin, y2 = x1 sin + x2 cos, cos / sin
//                  [seq, head_dim/2] f32 broadcast over batch and heads, arithmetic in f32, result in
//                  x's dtype; DSL twin Tyr/GPU/Kernels/Rotary.lean:13-66 (rotaryFwd, f32 64x64).
//   layernorm      Tyr/GPU/Kernels/FusedLayerNorm.lean:28-140 (tkFusedLayerNormResidual1024):
//                  out_resid = bf16(x + residual); statistics of the rounded out_resid in f32 over the
//                  whole row; out = bf16((r - mean) * rsqrt(var + eps) * weight + bias); expected
//                  values Examples/GPU/RunLayerNorm.lean:27-33 (torch layer_norm of x + residual).
//   decode append  Tyr/Model/Qwen/Attention.lean:172-196 (forwardStep): applyRotaryEmb on the
//                  single-token q and k, then sliceScatter of k and v into row `seq` of the
//                  [batch, kv_heads, maxLen, head_dim] cache.
//
// All four are bound by HBM bandwidth: every lane moves 16-byte pieces, consecutive lanes touch
// consecutive addresses, and the grids have many more workgroups than the device has CUs.
#include "common.hpp"
#include "launch.hpp"
#include <type_traits>

namespace tyr {

namespace rw {
constexpr int THREADS = 256;
constexpr int STREAM_THREADS = 64;      // one wave per workgroup for the pure streaming kernels

__device__ __forceinline__ void unpack8(u32x4 v, float (&f)[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) { f[2 * i] = bf16_lo(v[i]); f[2 * i + 1] = bf16_hi(v[i]); }
}
__device__ __forceinline__ u32x4 pack8(const float (&f)[8]) {
    u32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = pack_bf16(f[2 * i], f[2 * i + 1]);
    return v;
}

// Rotates one 16-byte piece pair: a = elements [e0, e0+E) of the first half, b = the same
// elements of the second half; c / s point at cos[e0], sin[e0].
template <typename T> struct Piece;
template <> struct Piece<float> {
    static constexpr int E = 4;
    static __device__ __forceinline__ void rotate(u32x4& a, u32x4& b, const float* c, const float* s) {
        const f32x4 cv = *reinterpret_cast<const f32x4*>(c), sv = *reinterpret_cast<const f32x4*>(s);
        f32x4 x1 = __builtin_bit_cast(f32x4, a), x2 = __builtin_bit_cast(f32x4, b), y1, y2;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma clang fp contract(off)   // separate multiplies and add, as the reference expression evaluates
            y1[i] = x1[i] * cv[i] - x2[i] * sv[i];
            y2[i] = x1[i] * sv[i] + x2[i] * cv[i];
        }
        a = __builtin_bit_cast(u32x4, y1);
        b = __builtin_bit_cast(u32x4, y2);
    }
};
template <> struct Piece<uint16_t> {                 // bf16
    static constexpr int E = 8;
    static __device__ __forceinline__ void rotate(u32x4& a, u32x4& b, const float* c, const float* s) {
        float x1[8], x2[8], y1[8], y2[8], cv[8], sv[8];
        unpack8(a, x1);
        unpack8(b, x2);
        *reinterpret_cast<f32x4*>(cv) = *reinterpret_cast<const f32x4*>(c);
        *reinterpret_cast<f32x4*>(cv + 4) = *reinterpret_cast<const f32x4*>(c + 4);
        *reinterpret_cast<f32x4*>(sv) = *reinterpret_cast<const f32x4*>(s);
        *reinterpret_cast<f32x4*>(sv + 4) = *reinterpret_cast<const f32x4*>(s + 4);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
#pragma clang fp contract(off)
            y1[i] = x1[i] * cv[i] - x2[i] * sv[i];
            y2[i] = x1[i] * sv[i] + x2[i] * cv[i];
        }
        a = pack8(y1);
        b = pack8(y2);
    }
};
}  // namespace rw

// ------------------------------------------------------------------------------------------
template <bool CACHED>
__global__ __launch_bounds__(rw::THREADS) void copy_kernel(const u32x4* __restrict__ src, u32x4* __restrict__ dst,
                                                           size_t n16, const unsigned char* __restrict__ src_tail,
                                                           unsigned char* __restrict__ dst_tail, int tail) {
    // One 16-byte piece per lane, one wave per workgroup, no loop: the dispatcher then walks the
    // buffers as one contiguous front (measured on a 1 GiB copy: 6.7 TB/s of read + write traffic,
    // against 6.0 for a grid-stride loop with four loads in flight per lane).
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n16) st_global_16_nt(dst + i, ld_stream_16<CACHED>(src + i));
    if (blockIdx.x == 0 && (int)threadIdx.x < tail) dst_tail[threadIdx.x] = src_tail[threadIdx.x];
}

// x, y: [B*S*H][D].  One thread rotates one piece pair; a row takes per_row = D / (2E) consecutive threads.  I = uint32_t
// unless there are more threads than that counts (x from 137 GB on): with 64-bit divisions a thread spent as long on its
// indices as on its 64 bytes (together with plain loads 2222 x 32 heads of 128: 8.4 -> 7.0 us, 36 MB).
template <typename T, bool CACHED, typename I>
__global__ __launch_bounds__(rw::THREADS) void rope_kernel(const T* __restrict__ x, const float* __restrict__ cosp,
                                                           const float* __restrict__ sinp, T* __restrict__ y,
                                                           I threads, unsigned S, unsigned H, unsigned per_row) {
    constexpr unsigned E = rw::Piece<T>::E;
    const I id = (I)blockIdx.x * rw::THREADS + threadIdx.x;
    if (id >= threads) return;
    const I row = id / per_row;
    const unsigned half = per_row * E, e0 = (unsigned)(id - row * per_row) * E;
    const unsigned s = (unsigned)(row / H % S);
    const size_t at = (size_t)row * 2 * half + e0;
    u32x4 a = ld_stream_16<CACHED>(x + at), b = ld_stream_16<CACHED>(x + at + half);
    rw::Piece<T>::rotate(a, b, cosp + (size_t)s * half + e0, sinp + (size_t)s * half + e0);
    st_global_16_nt(y + at, a);
    st_global_16_nt(y + at + half, b);
}

// Rows 0 .. B*Hq-1: q rows (rotated into q_out).  Then B*Hkv k rows (rotated into row `pos` of the
// k cache) and B*Hkv v rows (copied into row `pos` of the v cache).  cos / sin: [D/2] of position pos.
__global__ __launch_bounds__(rw::THREADS) void decode_rope_append_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k_new, const uint16_t* __restrict__ v_new,
    const float* __restrict__ cosp, const float* __restrict__ sinp, uint16_t* __restrict__ q_out,
    uint16_t* __restrict__ k_cache, uint16_t* __restrict__ v_cache, int nq, int nkv, int D, size_t kv_stride,
    size_t pos) {
    const int per_row = D / 16;
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    const int row = id / per_row;
    if (row >= nq + 2 * nkv) return;
    const int e0 = (id % per_row) * 8;
    const uint16_t* src;
    uint16_t* dst;
    bool rotate = true;
    if (row < nq) {
        src = q + (size_t)row * D;
        dst = q_out + (size_t)row * D;
    } else if (row < nq + nkv) {
        src = k_new + (size_t)(row - nq) * D;
        dst = k_cache + ((size_t)(row - nq) * kv_stride + pos) * D;
    } else {
        src = v_new + (size_t)(row - nq - nkv) * D;
        dst = v_cache + ((size_t)(row - nq - nkv) * kv_stride + pos) * D;
        rotate = false;
    }
    u32x4 a = ld_global_16(src + e0), b = ld_global_16(src + D / 2 + e0);
    if (rotate) rw::Piece<uint16_t>::rotate(a, b, cosp + e0, sinp + e0);
    st_global_16(dst + e0, a);
    st_global_16(dst + D / 2 + e0, b);
}

// WPR waves per row; a lane holds P <= 2 pieces (8 bf16) of it, lane, lane + 64 * WPR, so that all loads of a row, weights
// included, are under way at once and many waves share the chip (one wave per row, up to 16 pieces a lane: 2222 x 4096
// 16.8 us, 300 x 8192 17; so 13.1 and 7.1).
template <int WPR, int P, bool CACHED>
__global__ __launch_bounds__(WPR > 4 ? 64 * WPR : 256) void layernorm_residual_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ res, const uint16_t* __restrict__ weight,
    const uint16_t* __restrict__ bias, uint16_t* __restrict__ out, uint16_t* __restrict__ out_resid, size_t rows,
    int d_model, float eps) {
    constexpr int RPB = WPR > 4 ? 1 : 4 / WPR;
    __shared__ float2 part[RPB][WPR];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wr = wave % WPR;
    const size_t row = (size_t)blockIdx.x * RPB + wave / WPR;
    const bool live = row < rows;
    if (WPR == 1 && !live) return;
    const int pieces = live ? d_model / 8 : 0;
    const size_t at = row * d_model;
    float v[P][8];
    u32x4 a[P], b[P], w[P], bi[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int pc = lane + 64 * (wr + WPR * p);
        if (pc < pieces) {
            a[p] = ld_stream_16<CACHED>(x + at + pc * 8);
            b[p] = ld_stream_16<CACHED>(res + at + pc * 8);
        }
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int pc = lane + 64 * (wr + WPR * p);
        if (pc < pieces) {
            w[p] = ld_global_16(weight + pc * 8);
            bi[p] = ld_global_16(bias + pc * 8);
        }
    }
    float sum = 0.0f;
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int pc = lane + 64 * (wr + WPR * p);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[p][i] = 0.0f;
        if (pc < pieces) {
            float f[8], g[8];
            rw::unpack8(a[p], f);
            rw::unpack8(b[p], g);
#pragma unroll
            for (int i = 0; i < 8; ++i) f[i] += g[i];
            const u32x4 r16 = rw::pack8(f);                     // out_resid is the bf16-rounded sum ...
            st_global_16_nt(out_resid + at + pc * 8, r16);
            rw::unpack8(r16, v[p]);                             // ... and the statistics are taken from it
#pragma unroll
            for (int i = 0; i < 8; ++i) sum += v[p][i];
        }
    }
    auto wave_sum = [](float s) {
#pragma unroll
        for (int o = 1; o < 32; o <<= 1) s += __shfl_xor(s, o, 64);
        return sum_xor32(s);
    };
    // mean and sum of squares about it: of each wave's elements, then of the row's waves together
    auto elements = [&](int i) {                                // of wave i
        int c = 0;
#pragma unroll
        for (int p = 0; p < P; ++p) c += max(0, min(64, pieces - 64 * (i + WPR * p)));
        return 8.0f * (float)c;
    };
    float mean = wave_sum(sum) / fmaxf(elements(wr), 1.0f);
    float sq = 0.0f;
#pragma unroll
    for (int p = 0; p < P; ++p)
        if (lane + 64 * (wr + WPR * p) < pieces) {
#pragma unroll
            for (int i = 0; i < 8; ++i) { const float c = v[p][i] - mean; sq += c * c; }
        }
    sq = wave_sum(sq);
    if constexpr (WPR > 1) {
        if (lane == 0) part[wave / WPR][wr] = float2{mean, sq};
        __syncthreads();
        if (!live) return;
        float2 q[WPR];
        float total = 0.0f;
#pragma unroll
        for (int i = 0; i < WPR; ++i) {
            q[i] = part[wave / WPR][i];
            total += q[i].x * elements(i);
        }
        mean = total / (float)d_model;
        sq = 0.0f;
#pragma unroll
        for (int i = 0; i < WPR; ++i) { const float d = q[i].x - mean; sq += q[i].y + elements(i) * d * d; }
    }
    const float inv_std = rsqrtf(sq / (float)d_model + eps);
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int pc = lane + 64 * (wr + WPR * p);
        if (pc < pieces) {
            float wf[8], bf[8], o[8];
            rw::unpack8(w[p], wf);
            rw::unpack8(bi[p], bf);
#pragma unroll
            for (int i = 0; i < 8; ++i) o[i] = (v[p][i] - mean) * inv_std * wf[i] + bf[i];
            st_global_16_nt(out + at + pc * 8, rw::pack8(o));
        }
    }
}

// ------------------------------------------------------------------------------------------
int launch_copy(const void* src, void* dst, size_t bytes, hipStream_t stream) {
    const size_t n16 = bytes / 16;
    const int tail = (int)(bytes % 16);
    size_t blocks = (n16 + rw::STREAM_THREADS - 1) / rw::STREAM_THREADS;
    if (blocks == 0) blocks = 1;
    if (blocks > 0x7fffffffull) return -1;             // 2^31 workgroups of 1 KiB: 2 TiB
    launch_kernel((2 * bytes <= kStreamCached ? copy_kernel<true> : copy_kernel<false>), dim3((unsigned)blocks), dim3(rw::STREAM_THREADS), 0, stream,
                       static_cast<const u32x4*>(src), static_cast<u32x4*>(dst), n16,
                       static_cast<const unsigned char*>(src) + n16 * 16, static_cast<unsigned char*>(dst) + n16 * 16,
                       tail);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_rope_fwd(const void* x, const float* cosp, const float* sinp, void* y, size_t rows, int S, int H, int D,
                    int is_bf16, hipStream_t stream) {
    const unsigned per_row = D / (is_bf16 ? 16 : 8);
    const size_t threads = rows * per_row;
    auto go = [&](auto elem, auto cached, auto index) {
        using T = decltype(elem);
        using I = decltype(index);
        launch_kernel((rope_kernel<T, cached(), I>), dim3((unsigned)((threads + rw::THREADS - 1) / rw::THREADS)), dim3(rw::THREADS), 0,
                           stream, static_cast<const T*>(x), cosp, sinp, static_cast<T*>(y), (I)threads, (unsigned)S, (unsigned)H, per_row);
    };
    auto pick = [&](auto elem) {
        if (threads * 64 <= kStreamCached) go(elem, std::true_type{}, uint32_t{});
        else if (threads <= UINT32_MAX - rw::THREADS) go(elem, std::false_type{}, uint32_t{});
        else go(elem, std::false_type{}, size_t{});
    };
    if (is_bf16) pick(uint16_t{}); else pick(float{});
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_decode_rope_append(const void* q, const void* k_new, const void* v_new, const float* cosp,
                              const float* sinp, void* q_out, void* k_cache, void* v_cache, int B, int Hq, int Hkv,
                              int D, size_t kv_stride, size_t pos, hipStream_t stream) {
    const int nq = B * Hq, nkv = B * Hkv;
    const size_t threads = (size_t)(nq + 2 * nkv) * (D / 16);
    const size_t blocks = (threads + rw::THREADS - 1) / rw::THREADS;
    launch_kernel(decode_rope_append_kernel, dim3((unsigned)blocks), dim3(rw::THREADS), 0, stream,
                       static_cast<const uint16_t*>(q), static_cast<const uint16_t*>(k_new),
                       static_cast<const uint16_t*>(v_new), cosp, sinp, static_cast<uint16_t*>(q_out),
                       static_cast<uint16_t*>(k_cache), static_cast<uint16_t*>(v_cache), nq, nkv, D, kv_stride, pos);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_layernorm_residual(const void* x, const void* residual, const void* weight, const void* bias, void* out,
                              void* out_resid, size_t rows, int d_model, float eps, hipStream_t stream) {
    auto go = [&](auto wpr, auto p) {
        constexpr int W = wpr(), RPB = W > 4 ? 1 : 4 / W;       // rows per workgroup
        auto kernel = rows * d_model * 8 <= kStreamCached ? &layernorm_residual_kernel<W, p(), true> : &layernorm_residual_kernel<W, p(), false>;
        launch_kernel(kernel, dim3((unsigned)((rows + RPB - 1) / RPB)), dim3(W > 4 ? 64 * W : 256), 0, stream,
                           static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(residual), static_cast<const uint16_t*>(weight),
                           static_cast<const uint16_t*>(bias), static_cast<uint16_t*>(out), static_cast<uint16_t*>(out_resid), rows,
                           d_model, eps);
    };
    using std::integral_constant;
    if (d_model <= 512) go(integral_constant<int, 1>{}, integral_constant<int, 1>{});
    else if (d_model <= 1024) go(integral_constant<int, 1>{}, integral_constant<int, 2>{});
    else if (d_model <= 2048) go(integral_constant<int, 2>{}, integral_constant<int, 2>{});
    else if (d_model <= 4096) go(integral_constant<int, 4>{}, integral_constant<int, 2>{});
    else go(integral_constant<int, 8>{}, integral_constant<int, 2>{});
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace tyr
