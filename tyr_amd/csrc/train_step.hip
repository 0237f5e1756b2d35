// The element-wise half of the reference's attention train step (gfx950), fused into two streaming kernels.
//
// Reference semantics (Examples/GPU/RunMhaH100Train.lean:60-93, `oneKernelTrainStep`), which the reference
// evaluates as a chain of LibTorch element-wise calls around its forward and backward kernels:
//   lossAndGradOut  :60-67   diff = f32(out) - f32(target);  loss = 0.5 * mean(diff * diff);
//                            dO = bf16(diff / nElems)
//   sgdUpdate       :69-70   param' = param - (grad * lr)            (f32 master, grad = f32(bf16 gradient))
//   :83-85                   q = bf16(qM) ... at the top of the next step
// Here: one pass over out / target writes dO and per-workgroup partial sums of diff^2 (a second, single
// workgroup turns them into the loss; up to 2^15 elements one workgroup does both); one pass per parameter reads the f32 master and the bf16 gradient and
// writes the updated master together with its bf16 copy for the next step's kernels.  Both are bound by HBM
// bandwidth: 8- or 16-byte pieces per lane, consecutive lanes on consecutive addresses, no loop.
// Products and differences are evaluated as separate f32 operations (no fused multiply-add) and the division
// is a true division, so dO and the updated masters are bit-identical to the LibTorch chain.
#include "../../include/tyr_hip.h"

#include <limits.h>

#include "common.hpp"

namespace tyr {
namespace {

constexpr int THREADS = 256;

__device__ __forceinline__ void unpack8(u32x4 v, float (&f)[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) { f[2 * i] = bf16_lo(v[i]); f[2 * i + 1] = bf16_hi(v[i]); }
}

// dO of an 8-element piece; returns its sum of diff^2
__device__ __forceinline__ float mse_piece(u32x4 out, u32x4 target, uint16_t* d_out, float n_elems) {
    float o[8], t[8], d[8], acc = 0.0f;
    unpack8(out, o);
    unpack8(target, t);
    u32x4 g;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
#pragma clang fp contract(off)
        d[e] = o[e] - t[e];
        acc = acc + d[e] * d[e];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) g[e] = pack_bf16(d[2 * e] / n_elems, d[2 * e + 1] / n_elems);
    st_global_16_nt(d_out, g);
    return acc;
}

// one 8-element piece per lane; partial[blockIdx.x] = sum over the workgroup of diff^2
template <bool CACHED>
__global__ __launch_bounds__(THREADS) void mse_grad_kernel(const uint16_t* __restrict__ out, const uint16_t* __restrict__ target,
                                                           uint16_t* __restrict__ d_out, float* __restrict__ partial,
                                                           size_t pieces, float n_elems) {
    __shared__ float wave_sum[THREADS / 64];
    const size_t i = (size_t)blockIdx.x * THREADS + threadIdx.x;
    float acc = 0.0f;
    if (i < pieces) acc = mse_piece(ld_stream_16<CACHED>(out + 8 * i), ld_stream_16<CACHED>(target + 8 * i), d_out + 8 * i, n_elems);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) acc += __shfl_xor(acc, m, 64);
    if ((threadIdx.x & 63) == 0) wave_sum[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = (wave_sum[0] + wave_sum[1]) + (wave_sum[2] + wave_sum[3]);
}

__device__ __forceinline__ double workgroup_sum(double acc, double (&part)[16]) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) acc += __shfl_xor(acc, m, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = acc;
    __syncthreads();
    double s = 0.0;
    for (int w = 0; w < 16; ++w) s += part[w];
    return s;
}

// loss = 0.5 * (sum of the partials) / n, summed in double by one workgroup.  Latency is all it costs: four 16-byte loads
// of a lane are in flight at once (65536 partials: 17.6 us with one 4-byte load at a time).
typedef f32x4 f32x4_a4 __attribute__((aligned(4)));      // the caller's workspace is aligned to a float only
__global__ __launch_bounds__(1024) void mse_loss_kernel(const float* __restrict__ partial, size_t count, double n_elems,
                                                        float* __restrict__ loss) {
    __shared__ double part[16];
    double acc = 0.0;
    const size_t quads = count / 4;
    for (size_t i = threadIdx.x; i < quads; i += 4096) {
        f32x4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = i + 1024 * u < quads ? reinterpret_cast<const f32x4_a4*>(partial)[i + 1024 * u] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < 4; ++u) acc += ((double)v[u][0] + (double)v[u][1]) + ((double)v[u][2] + (double)v[u][3]);
    }
    if (threadIdx.x < count % 4) acc += (double)partial[4 * quads + threadIdx.x];
    const double s = workgroup_sum(acc, part);
    if (threadIdx.x == 0) *loss = (float)(0.5 * s / n_elems);
}

// Both of the above in one launch of one workgroup, for at most ONE_PASS pieces: a launch costs more host time than the one workgroup
// loses there (7.2 us a call with two launches; 4.9 at 2^12, 6.2 at 2^15 elements with one).
constexpr int ONE_PASS = 4096;
__global__ __launch_bounds__(1024) void mse_grad_loss_kernel(const uint16_t* __restrict__ out, const uint16_t* __restrict__ target,
                                                             uint16_t* __restrict__ d_out, float* __restrict__ loss, int pieces,
                                                             float n_elems) {
    __shared__ double part[16];
    constexpr int P = ONE_PASS / 1024;
    u32x4 o[P], t[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int i = min((int)threadIdx.x + 1024 * p, pieces - 1);
        o[p] = ld_global_16(out + 8 * (size_t)i);
        t[p] = ld_global_16(target + 8 * (size_t)i);
    }
    double acc = 0.0;
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int i = threadIdx.x + 1024 * p;
        if (i < pieces) acc += (double)mse_piece(o[p], t[p], d_out + 8 * (size_t)i, n_elems);
    }
    const double s = workgroup_sum(acc, part);
    if (threadIdx.x == 0) *loss = (float)(0.5 * s / (double)n_elems);
}

// param' = param - (f32(grad) * lr); optionally also bf16(param').  param_out may be param itself (the in-place update), so
// neither of the two is declared restrict; a lane stores only the elements it loaded.
template <bool CACHED>
__global__ __launch_bounds__(THREADS) void sgd_kernel(const float* param, const uint16_t* __restrict__ grad, float lr,
                                                      float* param_out, uint16_t* __restrict__ param_out_bf16,
                                                      size_t n) {
    // a wave's 512 elements as two runs of 256: every load and store instruction covers whole cache lines (a lane with 8
    // consecutive elements leaves half of every line to its next instruction: 277 us for 2^27 elements, so 253, 6.4 TB/s).
    const size_t base = ((size_t)blockIdx.x * (THREADS / 64) + (threadIdx.x >> 6)) * 512 + (threadIdx.x & 63) * 4;
    f32x4 p[2];
    u32x2 g[2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
        if (base + 256 * h < n) {
            p[h] = __builtin_bit_cast(f32x4, ld_stream_16<CACHED>(param + base + 256 * h));
            auto gp = reinterpret_cast<const u32x2*>(grad + base + 256 * h);
            g[h] = CACHED ? *gp : __builtin_nontemporal_load(gp);
        }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if (base + 256 * h >= n) return;
        f32x4 r;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma clang fp contract(off)
            const float step = (e & 1 ? bf16_hi(g[h][e >> 1]) : bf16_lo(g[h][e >> 1])) * lr;
            r[e] = p[h][e] - step;
        }
        __builtin_nontemporal_store(r, reinterpret_cast<f32x4*>(param_out + base + 256 * h));
        if (param_out_bf16 != nullptr)
            __builtin_nontemporal_store(u32x2{pack_bf16(r[0], r[1]), pack_bf16(r[2], r[3])},
                                        reinterpret_cast<u32x2*>(param_out_bf16 + base + 256 * h));
    }
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace
}  // namespace tyr

extern "C" {

size_t tyr_hip_mse_loss_grad_workspace_bytes(uint64_t n) {
    const uint64_t pieces = (n + 7) / 8;
    return (size_t)((pieces + tyr::THREADS - 1) / tyr::THREADS) * sizeof(float);
}

int tyr_hip_mse_loss_grad(const void* out, const void* target, void* d_out, float* loss, uint64_t n, void* workspace,
                          size_t workspace_bytes, void* stream) {
    using namespace tyr;
    if (!out || !target || !d_out || !loss) return TYR_HIP_ERR_NULL_POINTER;
    if (n == 0) return TYR_HIP_ERR_BAD_SHAPE;
    if (n % 8 != 0) return TYR_HIP_ERR_UNSUPPORTED;
    const uint64_t pieces = n / 8, blocks = (pieces + THREADS - 1) / THREADS;
    if (blocks > (uint64_t)INT_MAX) return TYR_HIP_ERR_BAD_SHAPE;
    if (!aligned16(out) || !aligned16(target) || !aligned16(d_out) || (reinterpret_cast<uintptr_t>(loss) & 3u))
        return TYR_HIP_ERR_MISALIGNED;
    if (!workspace || workspace_bytes < tyr_hip_mse_loss_grad_workspace_bytes(n)) return TYR_HIP_ERR_WORKSPACE;
    if (reinterpret_cast<uintptr_t>(workspace) & 3u) return TYR_HIP_ERR_MISALIGNED;
    auto s = static_cast<hipStream_t>(stream);
    if (pieces <= ONE_PASS) {
        launch_kernel(mse_grad_loss_kernel, dim3(1), dim3(1024), 0, s, static_cast<const uint16_t*>(out),
                           static_cast<const uint16_t*>(target), static_cast<uint16_t*>(d_out), loss, (int)pieces, (float)n);
        return hipGetLastError() == hipSuccess ? TYR_HIP_OK : TYR_HIP_ERR_LAUNCH;
    }
    float* partial = static_cast<float*>(workspace);
    launch_kernel((6 * n <= kStreamCached ? mse_grad_kernel<true> : mse_grad_kernel<false>), dim3((unsigned)blocks), dim3(THREADS), 0, s, static_cast<const uint16_t*>(out),
                       static_cast<const uint16_t*>(target), static_cast<uint16_t*>(d_out), partial, (size_t)pieces, (float)n);
    if (hipGetLastError() != hipSuccess) return TYR_HIP_ERR_LAUNCH;
    launch_kernel(mse_loss_kernel, dim3(1), dim3(1024), 0, s, partial, (size_t)blocks, (double)n, loss);
    return hipGetLastError() == hipSuccess ? TYR_HIP_OK : TYR_HIP_ERR_LAUNCH;
}

int tyr_hip_sgd_step(const float* param, const void* grad, float lr, float* param_out, void* param_out_bf16, uint64_t n,
                     void* stream) {
    using namespace tyr;
    if (!param || !grad || !param_out) return TYR_HIP_ERR_NULL_POINTER;
    if (n == 0) return TYR_HIP_ERR_BAD_SHAPE;
    if (n % 8 != 0) return TYR_HIP_ERR_UNSUPPORTED;
    const uint64_t pieces = n / 8, blocks = (pieces + THREADS - 1) / THREADS;
    if (blocks > (uint64_t)INT_MAX) return TYR_HIP_ERR_BAD_SHAPE;
    if (!aligned16(param) || !aligned16(grad) || !aligned16(param_out) || !aligned16(param_out_bf16))
        return TYR_HIP_ERR_MISALIGNED;
    launch_kernel((12 * n <= kStreamCached ? sgd_kernel<true> : sgd_kernel<false>), dim3((unsigned)blocks), dim3(THREADS), 0, static_cast<hipStream_t>(stream), param,
                       static_cast<const uint16_t*>(grad), lr, param_out, static_cast<uint16_t*>(param_out_bf16), (size_t)n);
    return hipGetLastError() == hipSuccess ? TYR_HIP_OK : TYR_HIP_ERR_LAUNCH;
}

}  // extern "C"
