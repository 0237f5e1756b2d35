// Shared device-side vocabulary for the gfx950 kernels: vector types, MFMA wrappers,
// bf16 packing, cross-lane helpers.  Wave size is 64 everywhere.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <tuple>

namespace tyr {

// Launch without the <<< >>> form's stack of launch configurations, which a kernel's host stub pushes to and pops from: 2.12 us
// of host time a launch, 2.40 with it (an entry point's whole call, median of 8 processes: copy 4.22 -> 4.00, gemm 4.15 -> 3.92).
template <class... P, class... A>
inline void launch_kernel(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t stream, A... a) {
    std::tuple<P...> values{static_cast<P>(a)...};
    std::apply([&](P&... v) {
        void* args[] = {&v...};
        (void)hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, args, lds, stream);
    }, values);
}

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(8))) int i32x8;

constexpr int kWave = 64;

// ---- MFMA (dense, f32 accumulate) -------------------------------------------------
// Operand layout facts used throughout (lane = l, wave64):
//   32x32x16 bf16 : A lane holds row  l%32, k = 8*(l/32)+[0,8) ; B lane holds col l%32, same k.
//                   D reg r (0..15)  <-> row 8*(r/4) + 4*(l/32) + r%4, col l%32.
//   16x16x32 bf16 : A lane holds row  l%16, k = 8*(l/16)+[0,8) ; B lane holds col l%16, same k.
//                   D reg r (0..3)   <-> row 4*(l/16) + r, col l%16.
//   32x32x64 fp8  : as 32x32x16 with 32 bytes of k per lane (k = 32*(l/32)+[0,32)).
// Only "A and B use the same k <-> (lane group, slot) map" matters for correctness of a
// product, so kernels are free to permute k as long as both operands agree.

__device__ __forceinline__ f32x16 mfma_32x32x16_bf16(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// Products in asm, for a kernel that fills the register file and says which half of it a result lives in: acc = accumulation
// registers, vgpr = ordinary ones (begin: the accumulator starts from 0 or c).  The compiler does not see a product in the asm, so
// the caller keeps two wait states between an ordinary write of a, b or c and the product, and between the product and any other instruction
// on its result 12 (32x32x16) or 8 (16x16x32), as the compiler does behind its own; products in between count.
__device__ __forceinline__ void mfma_32x32x16_bf16_acc(f32x16& c, bf16x8 a, bf16x8 b) {
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma_16x16x32_bf16_vgpr(f32x4& c, bf16x8 a, bf16x8 b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma_16x16x32_bf16_vgpr_begin(f32x4& d, bf16x8 a, bf16x8 b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma_16x16x32_bf16_vgpr_begin(f32x4& d, bf16x8 a, bf16x8 b, f32x4 c) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %3" : "=&v"(d) : "v"(a), "v"(b), "v"(c));
}
__device__ __forceinline__ f32x4 mfma_16x16x32_bf16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// FP8 E4M3 x E4M3 (format code 0 on both operands), scales fixed at 1 (unscaled encoding).
__device__ __forceinline__ f32x16 mfma_32x32x64_e4m3(i32x8 a, i32x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
}

// ---- bf16 packing -----------------------------------------------------------------
// Round-to-nearest-even f32 -> bf16 pair (v_cvt_pk_bf16_f32); lo goes to bits [15:0].
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    bf16x2 r = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ float bf16_lo(uint32_t u) { return __builtin_bit_cast(float, u << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t u) { return __builtin_bit_cast(float, u & 0xffff0000u); }

// ---- cross-lane -------------------------------------------------------------------
// Value held by lane l^32.  v_permlane32_swap exchanges lanes 32-63 of its first register with
// lanes 0-31 of its second; fed the same value twice, the partner's value is in the first
// result for the upper half-wave and in the second for the lower half-wave.  (Selecting per
// half also stays right if the compiler assigns both operands to one register, in which case
// either result holds the partner's value.)
__device__ __forceinline__ float xor32(float x) {
    uint32_t u = __builtin_bit_cast(uint32_t, x);
    u32x2 s = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    uint32_t other = (threadIdx.x & 32) ? s.x : s.y;
    return __builtin_bit_cast(float, other);
}
// Value held by lane l^16 (same construction with v_permlane16_swap on 16-lane rows).
__device__ __forceinline__ float xor16(float x) {
    uint32_t u = __builtin_bit_cast(uint32_t, x);
    u32x2 s = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    uint32_t other = (threadIdx.x & 16) ? s.x : s.y;
    return __builtin_bit_cast(float, other);
}
__device__ __forceinline__ float max_xor32(float x) { return fmaxf(x, xor32(x)); }
__device__ __forceinline__ float sum_xor32(float x) { return x + xor32(x); }
__device__ __forceinline__ float max_xor16(float x) { return fmaxf(x, xor16(x)); }
__device__ __forceinline__ float sum_xor16(float x) { return x + xor16(x); }

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// ---- 16-byte global / LDS moves ----------------------------------------------------
__device__ __forceinline__ u32x4 ld_global_16(const void* p) { return *reinterpret_cast<const u32x4*>(p); }
__device__ __forceinline__ u32x2 ld_global_8(const void* p) { return *reinterpret_cast<const u32x2*>(p); }
__device__ __forceinline__ void st_global_16(void* p, u32x4 v) { *reinterpret_cast<u32x4*>(p) = v; }
// Streaming variants (non-temporal hint) for data that is touched once: the lines are not kept in
// the caches at the expense of reusable data.  On the decode and copy kernels this alone is worth
// 10-30 % of the achieved HBM bandwidth.
__device__ __forceinline__ u32x4 ld_global_16_nt(const void* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
}
__device__ __forceinline__ void st_global_16_nt(void* p, u32x4 v) {
    __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(p));
}
// Loads of a streaming kernel (each byte read once).  Up to kStreamCached bytes moved by the launch, plain loads find what
// the kernels before left in the 256 MB last-level cache (LayerNorm of 2222 x 4096, 73 MB: 16.1 us non-temporal, 13.1 plain;
// SGD of 2^23 elements within a train step: 22 and 19); beyond, they only displace each other (268 MB: 45.4 and 47.3; SGD
// of 2^26: 149 and 161).  Stores are non-temporal at every size: the lines of plain ones are written back while the next
// kernel waits.
constexpr size_t kStreamCached = (size_t)160 << 20;
template <bool CACHED>
__device__ __forceinline__ u32x4 ld_stream_16(const void* p) { return CACHED ? ld_global_16(p) : ld_global_16_nt(p); }

__device__ __forceinline__ void st_global_8(void* p, u32x2 v) { *reinterpret_cast<u32x2*>(p) = v; }

// 8x8 transpose of 16-bit elements held as 8 rows of 4 dwords: out[c] holds column c
// (8 elements = 4 dwords, element r in half (r&1) of dword r/2).
__device__ __forceinline__ void transpose8x8_b16(const u32x4 (&in)[8], u32x4 (&out)[8]) {
#pragma unroll
    for (int c2 = 0; c2 < 4; ++c2) {      // column pair (2*c2, 2*c2+1) lives in dword c2 of every row
        u32x4 lo, hi;
#pragma unroll
        for (int j = 0; j < 4; ++j) {     // output dword j packs rows 2j, 2j+1
            uint32_t x0 = in[2 * j][c2], x1 = in[2 * j + 1][c2];
            lo[j] = __builtin_amdgcn_perm(x1, x0, 0x05040100u);   // [x0.lo16, x1.lo16]
            hi[j] = __builtin_amdgcn_perm(x1, x0, 0x07060302u);   // [x0.hi16, x1.hi16]
        }
        out[2 * c2] = lo;
        out[2 * c2 + 1] = hi;
    }
}

// Makes the compiler treat v as produced here: any load feeding it is waited for at this point
// (and not, conservatively, at its first use inside a loop that has other loads in flight).
__device__ __forceinline__ void pin_registers(bf16x8& v) {
    u32x4 u = __builtin_bit_cast(u32x4, v);
    asm volatile("" : "+v"(u));
    v = __builtin_bit_cast(bf16x8, u);
}

// ds_read_b64_tr_b8: transposing LDS read for bytes.  Within each block of 16 lanes, lane 8q+p
// receives byte p of the 8-byte pieces addressed by lanes q, q+2, q+4, ..., q+14 of the block.
__device__ __forceinline__ u32x2 ds_read_tr8(const void* lds_ptr) {
    typedef __attribute__((ext_vector_type(2))) int i32x2;
    const i32x2 v = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) i32x2*)(lds_ptr));
    return __builtin_bit_cast(u32x2, v);
}

// Buffer resource (V#) for raw byte-addressed access to [base, base + bytes): loads beyond the
// range return zero.  On gfx950 the range check covers the whole offset, per-lane, scalar and immediate
// parts together (probed with a 4 KiB descriptor inside a larger allocation: a scalar offset of 4000
// gives data to the lanes below byte 4096 and zeros to the rest), so a slice index carried in the
// scalar offset is zero-filled past the end like a row index carried in the per-lane offset.
__device__ __forceinline__ u32x4 make_raw_rsrc(const void* base, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    return u32x4{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, bytes, 0x00020000u};
}

// 16 bytes per lane from global memory straight into LDS: lane i of the wave writes
// lds_base + 16 i (lds_base wave-uniform); the source is rsrc.base + voffset + soffset.
// Issued as opaque asm so that the compiler does not order later LDS reads behind it; the
// caller waits with wait_vmcnt0() (and a barrier) before anyone reads the destination.  M0 is
// written here.  M0 is a reserved register for this compiler (it never holds a value across
// statements; the compiler writes it right before each of its own instructions that read it, and
// hipcc rejects it on a clobber list with a warning), so the write cannot corrupt compiler state as
// long as no compiler-generated M0 reader sits between its own write and use -- which
// tests/test_m0_discipline.py checks on the assembly of every kernel file that includes this one:
// the only M0 accesses are these writes, each followed by the LDS-DMA loads that consume it.
__device__ __forceinline__ void load_global_to_lds_16(u32x4 rsrc, uint32_t lds_base, int voffset, int soffset) {
    asm volatile(
        "s_mov_b32 m0, %0\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %1, %2, %3 offen lds"
        :
        : "s"(lds_base), "v"(voffset), "s"(rsrc), "s"(soffset)
        : "memory");
}
// N consecutive kilobytes of LDS from one M0 write: the instruction's immediate offset advances the
// LDS destination and the global source together, so request m uses immediate 1024 m and a per-lane
// offset that has 1024 m taken off (voffset_less[m] = source offset of request m - 1024 m >= 0).
template <int N>
__device__ __forceinline__ void load_global_to_lds_16xN(u32x4 rsrc, uint32_t lds_base, const int (&voffset_less)[N], int soffset) {
    static_assert(N == 1 || N == 2 || N == 4, "1, 2 or 4 requests per call");
    if constexpr (N == 1) {
        load_global_to_lds_16(rsrc, lds_base, voffset_less[0], soffset);
    } else if constexpr (N == 4) {
        asm volatile(
            "s_mov_b32 m0, %0\n\t"
            "s_nop 0\n\t"
            "buffer_load_dwordx4 %1, %5, %6 offen lds\n\t"
            "buffer_load_dwordx4 %2, %5, %6 offen offset:1024 lds\n\t"
            "buffer_load_dwordx4 %3, %5, %6 offen offset:2048 lds\n\t"
            "buffer_load_dwordx4 %4, %5, %6 offen offset:3072 lds"
            :
            : "s"(lds_base), "v"(voffset_less[0]), "v"(voffset_less[1]), "v"(voffset_less[2]), "v"(voffset_less[3]),
              "s"(rsrc), "s"(soffset)
            : "memory");
    } else {
        asm volatile(
            "s_mov_b32 m0, %0\n\t"
            "s_nop 0\n\t"
            "buffer_load_dwordx4 %1, %3, %4 offen lds\n\t"
            "buffer_load_dwordx4 %2, %3, %4 offen offset:1024 lds"
            :
            : "s"(lds_base), "v"(voffset_less[0]), "v"(voffset_less[1]), "s"(rsrc), "s"(soffset)
            : "memory");
    }
}
__device__ __forceinline__ void wait_vmcnt0() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// ds_read_b64_tr_b16: transposing LDS read.  Within each block of 16 lanes, lane 4q+p receives
// element p (16 bits) of the 8-byte pieces addressed by lanes q, q+4, q+8, q+12 of the block.
__device__ __forceinline__ bf16x4 ds_read_tr16(const void* lds_ptr) {
    typedef __attribute__((ext_vector_type(4))) short s16x4;
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4*)(lds_ptr));
    return __builtin_bit_cast(bf16x4, v);
}

// Epilogue of the 256x256-tile GEMMs: one wave's 128x128 f32 accumulator quadrant (4x4 MFMA tiles
// computed with the B fragment as row operand: lane = m row l%32, register e <-> n = 8(e/4) +
// 4(l/32) + e%4) goes to global memory as bf16 rows.  Each 32-row band passes through a private
// LDS scratch (32 rows x 272 B) so that the global stores are 16 bytes per lane along rows.
constexpr int kEpilogueScratchBytes = 32 * 272;
// rows / cols = how much of the 128x128 quadrant lies inside C (cols a multiple of 8).
// NJ = 32-column tiles of the wave's block (4: a 128x128 quadrant; 2: 128x64).
template <int NJ>
__device__ __forceinline__ void store_quadrant_bf16(const f32x16 (&acc)[4][NJ], float scale, unsigned char* scratch,
                                                    uint16_t* c_quadrant, int ldc, int lane, int rows, int cols) {
    const int r = lane & 31, g = lane >> 5;
    constexpr int CH = NJ * 4;                           // 16-byte chunks per row of the block
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                u32x2 v;
                v.x = pack_bf16(acc[i][j][q4 * 4 + 0] * scale, acc[i][j][q4 * 4 + 1] * scale);
                v.y = pack_bf16(acc[i][j][q4 * 4 + 2] * scale, acc[i][j][q4 * 4 + 3] * scale);
                *reinterpret_cast<u32x2*>(scratch + r * 272 + (j * 32 + q4 * 8 + g * 4) * 2) = v;
            }
#pragma unroll
        for (int k = 0; k < 32 * CH / 64; ++k) {
            const int row = lane / CH + (64 / CH) * k;
            const u32x4 v = *reinterpret_cast<const u32x4*>(scratch + row * 272 + (lane % CH) * 16);
            if (i * 32 + row < rows && (lane % CH) * 8 < cols)
                st_global_16(c_quadrant + (size_t)(i * 32 + row) * ldc + (lane % CH) * 8, v);
        }
    }
}

// Four f32 to e4m3, round to nearest even, saturating at +-448; NaN stays.
__device__ __forceinline__ uint32_t pack_e4m3(f32x4 v) {
#pragma unroll
    for (int x = 0; x < 4; ++x) v[x] = v[x] != v[x] ? v[x] : fminf(fmaxf(v[x], -448.0f), 448.0f);
    const int w = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], 0, false);
    return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], w, true);
}
// Epilogue variants of the fp8 GEMM beyond "one scalar, bf16 out": per-row and per-column scales and the
// output element type.  The common case (no vectors, bf16) takes store_quadrant_bf16 above.
struct GemmEpilogue {
    float scale;                 // multiplies every element
    const float* row_scale;      // [M] or nullptr
    const float* col_scale;      // [N] or nullptr
    int out;                     // 0 = bf16, 1 = f32, 2 = e4m3 (round to nearest even, saturating at +-448)
    __device__ __host__ bool plain_bf16() const { return out == 0 && row_scale == nullptr && col_scale == nullptr; }
};
// Four scaled elements of C (row pitch N) from column gn on.
__device__ __forceinline__ void store_scaled4(const GemmEpilogue& ep, void* C, int N, int gm, int gn, f32x4 v) {
    const size_t at = (size_t)gm * N + gn;
    if (ep.out == 1) {
        *reinterpret_cast<f32x4*>(static_cast<float*>(C) + at) = v;
    } else if (ep.out == 2) {
        *reinterpret_cast<uint32_t*>(static_cast<uint8_t*>(C) + at) = pack_e4m3(v);
    } else {
        st_global_8(static_cast<uint16_t*>(C) + at, u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])});
    }
}
// One wave's 128x128 accumulator quadrant (layout as in store_quadrant_bf16) written straight from registers:
// a lane stores the 4 consecutive n of a register group of its row.  gm0 / gn0 = global row / column of the
// quadrant's first element; M, N = extents of C (row pitch N elements).
__device__ __forceinline__ void store_quadrant_ex(const f32x16 (&acc)[4][4], const GemmEpilogue& ep, void* C, int M, int N,
                                                  int gm0, int gn0, int lane) {
    const int r = lane & 31, g = lane >> 5;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int gm = gm0 + i * 32 + r;
        if (gm >= M) continue;
        const float rs = ep.scale * (ep.row_scale ? ep.row_scale[gm] : 1.0f);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                const int gn = gn0 + j * 32 + q4 * 8 + g * 4;
                if (gn >= N) continue;                       // N is a multiple of 16: a group of 4 is inside or outside
                f32x4 v = f32x4{acc[i][j][q4 * 4], acc[i][j][q4 * 4 + 1], acc[i][j][q4 * 4 + 2], acc[i][j][q4 * 4 + 3]} * rs;
                if (ep.col_scale) v *= *reinterpret_cast<const f32x4*>(ep.col_scale + gn);
                store_scaled4(ep, C, N, gm, gn, v);
            }
    }
}
// One wave's 128x64 block the same way, but through the wave's LDS scratch: each 32-row band as f32 (rows of 64 + 4), read back
// along the rows, so that a store is 16 bytes a lane and whole rows of the block (64 to 256 bytes) whatever the element, and
// the row and column scales are read once a lane.  Straight from registers a store touches 64 lines: M = 1065, N = 7136,
// K = 448 bf16 out 20.9 us, 12.2 this way (11.0 without vectors); 4096^3 60.5 -> 51.0, 8192^3 402 -> 375.
template <int OUT>
__device__ __forceinline__ void store_block_scaled(const f32x16 (&acc)[4][2], const GemmEpilogue& ep, unsigned char* scratch, void* C,
                                                   int M, int N, int gm0, int gn0, int lane) {
    constexpr int ES = OUT == 0 ? 2 : OUT == 1 ? 4 : 1, W = 16 / ES, LPR = 64 / W;      // columns a lane, lanes a row
    const int r = lane & 31, g = lane >> 5;
    const int gn = gn0 + (lane % LPR) * W;                   // N is a multiple of 16: inside or outside as a whole
    float rs[4];
    f32x4 cs[W / 4];
#pragma unroll
    for (int i = 0; i < 4; ++i) rs[i] = ep.scale * (ep.row_scale ? ep.row_scale[min(gm0 + i * 32 + r, M - 1)] : 1.0f);
#pragma unroll
    for (int x = 0; x < W / 4; ++x)
        cs[x] = ep.col_scale && gn < N ? *reinterpret_cast<const f32x4*>(ep.col_scale + gn + 4 * x) : f32x4{1.0f, 1.0f, 1.0f, 1.0f};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4)
                *reinterpret_cast<f32x4*>(scratch + r * 272 + (j * 32 + q4 * 8 + g * 4) * 4) =
                    f32x4{acc[i][j][q4 * 4], acc[i][j][q4 * 4 + 1], acc[i][j][q4 * 4 + 2], acc[i][j][q4 * 4 + 3]} * rs[i];
#pragma unroll
        for (int k = 0; k < 32 / W; ++k) {
            const int row = lane / LPR + W * k, gm = gm0 + i * 32 + row;
            const unsigned char* from = scratch + row * 272 + (lane % LPR) * (W * 4);
            u32x4 out;
            if constexpr (OUT == 1) {
                out = __builtin_bit_cast(u32x4, *reinterpret_cast<const f32x4*>(from) * cs[0]);
            } else {
#pragma unroll
                for (int x = 0; x < W / 4; ++x) {
                    const f32x4 v = *reinterpret_cast<const f32x4*>(from + 16 * x) * cs[x];
                    if constexpr (OUT == 0) {
                        out[2 * x] = pack_bf16(v[0], v[1]);
                        out[2 * x + 1] = pack_bf16(v[2], v[3]);
                    } else {
                        out[x] = pack_e4m3(v);
                    }
                }
            }
            if (gm < M && gn < N) st_global_16(static_cast<unsigned char*>(C) + ((size_t)gm * N + gn) * ES, out);
        }
    }
}

// Grid remap for the 8 XCDs of an MI355X: consecutive workgroup ids are dealt round-robin
// to the XCDs, each with its own L2.  This returns a logical id such that the workgroups
// that land on one XCD cover one contiguous range of logical ids (so neighbours in the
// logical order share an L2).  Falls back to the identity when n is not a multiple of 8.
__device__ __forceinline__ uint32_t xcd_remap(uint32_t pid, uint32_t n) {
    if (n % 8u) return pid;
    return (pid % 8u) * (n / 8u) + pid / 8u;
}

// What an attention launch masks besides the causal rule: nothing, lengths and / or a window, or a key mask.
enum class AttnMask { None, Limits, Keys };

// ---- key mask: the 64-key tiles among keys [0, end) that hold a visible one lie in [first, last) ------------------
// Read from both ends, 8 tiles an end and round (one byte a lane and tile, all 16 loads in flight), until a visible key is
// met: one memory latency where nothing is hidden at the ends, and a padded batch's empty tiles cost 1/8 of one each
// instead of a step of the attention loop (1 us).  end >= 1; nothing visible: first == last.
struct TileSpan { int first, last; };
__device__ __forceinline__ TileSpan visible_tiles(const uint8_t* mask, int end, int lane) {
    constexpr int AT_ONCE = 8;
    TileSpan s{0, (end + 63) / 64};
    bool front = false, back = false;
    while (s.first < s.last && !(front && back)) {
        uint8_t f[AT_ONCE], b[AT_ONCE];
#pragma unroll
        for (int u = 0; u < AT_ONCE; ++u) {
            f[u] = mask[min((s.first + u) * 64 + lane, end - 1)];
            b[u] = mask[max(0, min((s.last - 1 - u) * 64 + lane, end - 1))];
        }
        uint32_t in_front = 0, in_back = 0;
#pragma unroll
        for (int u = 0; u < AT_ONCE; ++u) {
            in_front |= (uint32_t)(__builtin_amdgcn_ballot_w64(f[u] != 0) != 0) << u;
            in_back |= (uint32_t)(__builtin_amdgcn_ballot_w64(b[u] != 0) != 0) << u;
        }
        if (!front) {
            front = in_front != 0;
            s.first = front ? s.first + __builtin_ctz(in_front) : min(s.first + AT_ONCE, s.last);
        }
        if (!back) {
            back = in_back != 0;
            s.last = back ? s.last - __builtin_ctz(in_back) : max(s.last - AT_ONCE, s.first);
        }
    }
    return {__builtin_amdgcn_readfirstlane(s.first), __builtin_amdgcn_readfirstlane(max(s.first, s.last))};
}

// ---- order of the query tiles of an attention launch ---------------------------------------------------------
// A launch has one job per (query head, tile rank); rank 0 is the longest causal tile.  Consecutive workgroup ids go to the
// 8 XCDs in turn, and of the ids an XCD gets, id i and id i + 32 share a CU (two workgroups fit).
//   paired (causal, many jobs): a job is the tiles ntq-1-rank and rank one after the other, so all jobs are equal; group
//     by group, so that the jobs that share a K / V run together.
//   single (few jobs): one tile per job, longest first -- and the first 32 of an XCD in ascending order, so that the
//     second workgroup of a CU is the longer the shorter its first one is.
// With grouped queries the unit dealt to an XCD is a (batch, kv head) group, whose G heads share one K / V.
struct AttnOrder {
    int BH, Hq, G, ntr, single;                      // ntr = ranks per head
    __host__ __device__ __forceinline__ void decode(int id, int& bh, int& rank, int& kvbh) const {
        const int ngroups = BH / G, hkv = Hq / G;
        if ((ngroups & 7) == 0) {
            const int xcd = id & 7, heads = BH >> 3;
            int slot = id >> 3, head;
            if (single) {
                if (slot < 32 && heads * ntr > 32) slot = 31 - slot;
                rank = slot / heads;
                const int r = slot % heads;
                kvbh = (r / G) * 8 + xcd;
                head = r % G;
            } else {
                const int per_group = G * ntr, within = slot % per_group;
                kvbh = (slot / per_group) * 8 + xcd;
                rank = within / G;
                head = within % G;
            }
            bh = (kvbh / hkv) * Hq + (kvbh % hkv) * G + head;
        } else {
            if (single) {
                if (id < 256 && BH * ntr > 256) id = 255 - id;
                rank = id / BH;
                bh = id % BH;
            } else {
                bh = id / ntr;
                rank = id % ntr;
            }
            kvbh = (bh / Hq) * hkv + (bh % Hq) / G;
        }
    }
};
// What one job of a launch is: `rows` query rows (128, or 64 with the keys of every tile shared by two waves), and for
// causal launches paired tiles or single ones.  dq: for the dQ kernel, whose steps take other times than the forward's.
struct AttnShape { int rows, pair, single; };
AttnShape attn_shape(int64_t bh, int N, int D, bool causal, int window, bool dq);
double attn_us(int64_t bh, int N, int D, bool causal, int window, bool dq);      // its launch, estimated

}  // namespace tyr
