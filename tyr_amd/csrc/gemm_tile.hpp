// Small and medium GEMM tiles for gfx950, bf16 and fp8 (OCP E4M3): C = epilogue(A B), A [M,K], B [K,N] or [N,K].
//
// The 256x256-tile kernels of gemm_bf16.hip / gemm_fp8.hip need 256 output tiles to fill the device; a product with
// fewer leaves CUs idle, and with one workgroup per CU every K slice costs a full memory latency.  Here the tile is
// small and the K range is shared out instead: the waves of a workgroup form KG k-groups, group kg takes the 128-byte
// pieces kg, kg + KG, ... of every operand row, and the groups' f32 accumulators are added in LDS at the end (a fixed
// order, so results are reproducible).  Where even that leaves CUs idle (few tiles, long K) the K range is also split
// over workgroups: each writes an f32 partial and gemm_tile_reduce_kernel adds them.
//
// What bounds it: bytes into the CU.  A workgroup moves (BM + BN) * K bytes-per-element bytes for BM * BN * K
// products; L2-resident operands arrive at 54 B/clk and CU by LDS-DMA (measured; fragment-shaped loads straight into
// registers, 16 rows x 64 B per instruction, only reach 16 B/clk, which is why everything goes through LDS), and from
// HBM at 6-6.5 TB/s in all.  So tiles are as large as the number of workgroups allows, and each wave keeps several
// pieces in flight: its requests are awaited with counted s_waitcnt, never drained inside the loop.
//
// LDS: one ring of ST stages per k-group; a stage holds BM rows x 128 B of A and 128 B-deep B (BN rows x 128 B, or
// 128 / ES rows x BN * ES bytes of a [K,N] B), 16-byte chunks XOR-swizzled so that fragment reads are conflict-free.
// A k-group of one wave owns its ring alone and needs no barrier; otherwise one barrier per piece.
#pragma once
#include <limits.h>
#include <math.h>

#include "common.hpp"

namespace tyr {
namespace gt {

constexpr int KB = 128;                              // bytes of every operand row per piece

template <int ES_, bool TB_, int BM_, int BN_, int WTM_, int WTN_, int KG_, int ST_>
struct Cfg {
    static constexpr int ES = ES_;                   // bytes per element: 2 = bf16, 1 = e4m3
    static constexpr bool TB = TB_;                  // B is [N,K]
    static constexpr int BM = BM_, BN = BN_, WTM = WTM_, WTN = WTN_, KG = KG_, ST = ST_;
    static constexpr int MF = (WTM % 32 == 0 && WTN % 32 == 0) ? 32 : 16;      // MFMA tile edge
    static constexpr int MT = WTM / MF, NT = WTN / MF;
    static constexpr int WPG = (BM / WTM) * (BN / WTN);                        // waves per k-group
    static constexpr int WAVES = WPG * KG, THREADS = 64 * WAVES;
    static constexpr int KS = ES == 2 ? MF / 8 : MF / 16;                      // MFMA k-steps per piece
    static constexpr int RA = BM / 8 / WPG, RB = BN / 8 / WPG;                 // 1 KiB requests per wave and piece
    static constexpr int STAGE = (BM + BN) * KB;
    static constexpr int RED_PITCH = BN + 4;                                   // floats; + 4 spreads rows over the banks
    static constexpr int RING = KG * ST * STAGE, RED = KG * BM * RED_PITCH * 4;
    static constexpr int LDS = RING > RED ? RING : RED;
    static constexpr int B_ROW = TB ? KB : BN * ES;                            // bytes per LDS row of B
    static_assert(BM % (8 * WPG) == 0 && BN % (8 * WPG) == 0, "whole requests per wave");
    static_assert(LDS <= 160 * 1024, "LDS of a CU");
    static_assert(WPG == 1 || ST >= 2, "a shared stage is refilled while the next is read");
};

// chunk (16 B) c of a row -> stored position.  Rows of 128 B: 16 consecutive rows put one chunk on all 64 banks.
__device__ __forceinline__ int swz_rows(int row, int c) { return c ^ ((row >> 1) & 7); }
// [K,N] B: what one half-wave of a transposing read touches (rows of one chunk group: 4 (b16) or 8 (b8) consecutive k, for
// 16-wide tiles of two k groups) must spread over the 256 B of the banks, whatever part of them one row covers.
template <class C>
__device__ __forceinline__ int swz_kn(int krow, int c) {
    constexpr int P = C::B_ROW;                      // 32, 64, 128 or 256 bytes
    if constexpr (C::ES == 2) {
        const int lo = krow & 3, grp = (krow >> 3) & 1;
        if constexpr (C::MF == 16) {                 // 8 rows x 32 B
            constexpr int SH = P >= 256 ? 0 : P >= 128 ? 1 : 2;      // row bits the pitch already spreads
            return c ^ (((lo >> SH) | (grp << (2 - SH))) << 1);
        } else {                                     // 4 rows x 64 B
            constexpr int SH = P >= 256 ? 0 : P >= 128 ? 1 : 2;
            return c ^ ((lo >> SH) << 2);
        }
    } else {
        const int lo = krow & 7, grp = (krow >> 5) & 1;
        constexpr int SH = P >= 256 ? 0 : P >= 128 ? 1 : P >= 64 ? 2 : 3;
        if constexpr (C::MF == 16) return c ^ ((lo >> SH) | (grp << (3 - SH)));      // 16 rows x 16 B
        else                       return c ^ ((lo >> SH) << 1);                     // 8 rows x 32 B
    }
}

// N kilobytes of LDS from N requests; voff[m] carries the -1024 (m % 4) of the immediate offsets
template <int N>
__device__ __forceinline__ void request(u32x4 rsrc, uint32_t dst, const int (&voff)[N], int soff) {
#pragma unroll
    for (int i = 0; i < N / 4; ++i) {
        const int four[4] = {voff[4 * i], voff[4 * i + 1], voff[4 * i + 2], voff[4 * i + 3]};
        load_global_to_lds_16xN<4>(rsrc, dst + 4096u * i, four, soff);
    }
    constexpr int DONE = N / 4 * 4;
    if constexpr (N % 4 >= 2) {
        const int two[2] = {voff[DONE], voff[DONE + 1]};
        load_global_to_lds_16xN<2>(rsrc, dst + 1024u * DONE, two, soff);
    }
    if constexpr (N % 2 == 1) {                      // the odd one is request 0 or 2 of its four: its own M0, no immediate
        const int one[1] = {voff[N - 1] + 1024 * ((N - 1) & 3)};
        load_global_to_lds_16xN<1>(rsrc, dst + 1024u * (N - 1), one, soff);
    }
}

template <int MF, int ES> struct Frag;
template <> struct Frag<32, 2> { typedef bf16x8 op; typedef f32x16 acc; };
template <> struct Frag<16, 2> { typedef bf16x8 op; typedef f32x4 acc; };
template <> struct Frag<32, 1> { typedef i32x8 op; typedef f32x16 acc; };
template <> struct Frag<16, 1> { typedef i32x8 op; typedef f32x4 acc; };
__device__ __forceinline__ f32x16 mma(bf16x8 a, bf16x8 b, f32x16 c) { return mfma_32x32x16_bf16(a, b, c); }
__device__ __forceinline__ f32x4 mma(bf16x8 a, bf16x8 b, f32x4 c) { return mfma_16x16x32_bf16(a, b, c); }
__device__ __forceinline__ f32x16 mma(i32x8 a, i32x8 b, f32x16 c) { return mfma_32x32x64_e4m3(a, b, c); }
__device__ __forceinline__ f32x4 mma(i32x8 a, i32x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
}
__device__ __forceinline__ i32x8 join(u32x4 a, u32x4 b) {
    return i32x8{(int)a.x, (int)a.y, (int)a.z, (int)a.w, (int)b.x, (int)b.y, (int)b.z, (int)b.w};
}

// four consecutive columns of C at (gm, gn), N % 4 == 0
__device__ __forceinline__ void store4(const GemmEpilogue& ep, void* C, int N, int gm, int gn, f32x4 v) {
    v *= ep.scale * (ep.row_scale ? ep.row_scale[gm] : 1.0f);
    if (ep.col_scale) v *= *reinterpret_cast<const f32x4*>(ep.col_scale + gn);
    store_scaled4(ep, C, N, gm, gn, v);
}

// Consecutive workgroup ids go round-robin to the 8 XCDs; this gives every XCD one contiguous range of logical ids.
__device__ __forceinline__ uint32_t xcd_range(uint32_t pid, uint32_t n) {
    const uint32_t x = pid & 7u, q = n >> 3, rem = n & 7u;
    return x * q + min(x, rem) + (pid >> 3);
}

}  // namespace gt

// Grid: x = tiles_m * tiles_n * splits, y = batch entry.  pieces = ceil(K * ES / 128); split z takes the pieces
// [z * pieces_per_split, ...).  With splits > 1 the tile goes to part[(z * batch + entry)][M][N] as f32.
template <class C>
__global__ __launch_bounds__(C::THREADS, (160 * 1024 / C::LDS) >= 2 ? 2 : 1) void gemm_tile_kernel(
    const unsigned char* __restrict__ A, const unsigned char* __restrict__ B, unsigned char* __restrict__ Cp, float* __restrict__ part,
    int M, int N, int K, int tiles_m, int tiles_n, int group_m, int splits, int pieces, int pieces_per_split, long stride_a, long stride_b,
    long stride_c, GemmEpilogue ep) {
    using namespace gt;
    typedef typename Frag<C::MF, C::ES>::op op_t;
    typedef typename Frag<C::MF, C::ES>::acc acc_t;
    constexpr int ES = C::ES, MF = C::MF;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    A += (size_t)blockIdx.y * stride_a * ES;
    B += (size_t)blockIdx.y * stride_b * ES;

    const int t = threadIdx.x;
    const int lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int kg = w / C::WPG, wg = w % C::WPG;      // k-group, wave within it
    const int wm = wg / (C::BN / C::WTN), wn = wg % (C::BN / C::WTN);

    // An XCD takes a contiguous range of ids, i.e. (split, then bands of group_m tile rows, then columns of a band): a
    // patch of tiles about as high as wide, so that few rows of A and columns of B pass through its L2.
    const uint32_t id = xcd_range(blockIdx.x, gridDim.x);
    const uint32_t tiles = (uint32_t)tiles_m * (uint32_t)tiles_n;
    const int z = (int)(id / tiles);
    const uint32_t in_z = id % tiles, band = in_z / ((uint32_t)group_m * tiles_n), in_band = in_z % ((uint32_t)group_m * tiles_n);
    const uint32_t rows = min((uint32_t)group_m, (uint32_t)tiles_m - band * group_m);
    const int tm = (int)(band * group_m + in_band % rows), tn = (int)(in_band / rows);
    const int m0 = tm * C::BM, n0 = tn * C::BN;

    // ---- requests.  A (and a [N,K] B): 8 rows x 128 B per request.  [K,N] B: 1024 / B_ROW k rows per request.
    // The immediate offsets 1024 (m % 4) move LDS destination and source together, so they are taken off the
    // per-lane offsets; descriptors start 3 KiB early so that those never go negative.  Rows past the end and
    // chunks past K read as zero (offset 2^31 is beyond every descriptor).
    const size_t row_bytes = (size_t)K * ES;
    const u32x4 a_rsrc = make_raw_rsrc(A + (size_t)m0 * row_bytes - 3072, (uint32_t)((size_t)min(M - m0, C::BM) * row_bytes) + 3072u);
    const u32x4 b_rsrc = C::TB
        ? make_raw_rsrc(B + (size_t)n0 * row_bytes - 3072, (uint32_t)((size_t)min(N - n0, C::BN) * row_bytes) + 3072u)
        : make_raw_rsrc(B + (size_t)n0 * ES - 3072, (uint32_t)min(((size_t)K * N - n0) * ES + 3072, (size_t)0xffffffffu));
    int a_voff[C::RA], b_voff[C::RB];
    int a_chunk[C::RA], b_chunk[C::RB];              // logical chunk of this lane's 16 bytes (K tail)
#pragma unroll
    for (int m = 0; m < C::RA; ++m) {
        const int row = (wg * C::RA + m) * 8 + (lane >> 3);
        a_chunk[m] = swz_rows(row, lane & 7);
        a_voff[m] = row * (int)row_bytes + a_chunk[m] * 16 + 3072 - 1024 * (m & 3);
    }
#pragma unroll
    for (int m = 0; m < C::RB; ++m) {
        if (C::TB) {
            const int row = (wg * C::RB + m) * 8 + (lane >> 3);
            b_chunk[m] = swz_rows(row, lane & 7);
            b_voff[m] = row * (int)row_bytes + b_chunk[m] * 16 + 3072 - 1024 * (m & 3);
        } else {
            constexpr int CPR = C::B_ROW / 16;       // chunks per k row
            const int krow = (wg * C::RB + m) * (64 / CPR) + lane / CPR;
            b_chunk[m] = 0;
            b_voff[m] = krow * N * ES + swz_kn<C>(krow, lane % CPR) * 16 + 3072 - 1024 * (m & 3);
        }
    }
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
    const uint32_t ring = __builtin_amdgcn_readfirstlane(lds_base + (uint32_t)kg * (C::ST * C::STAGE));
    const int p0 = z * pieces_per_split;
    const int np = min(pieces, p0 + pieces_per_split) - p0;          // pieces of this workgroup
    const int n_own = np > kg ? (np - kg + C::KG - 1) / C::KG : 0;   // pieces of this k-group
    auto issue = [&](int i, int st) {
        const int p = p0 + kg + i * C::KG;
        const int a_soff = p * KB;
        const int b_soff = C::TB ? p * KB : p * (KB / ES) * N * ES;
        const uint32_t dst = ring + (uint32_t)st * C::STAGE;
        int av[C::RA], bv[C::RB];
        const int chunks = ((int)row_bytes - p * KB) >> 4;           // chunks of this piece inside K
#pragma unroll
        for (int m = 0; m < C::RA; ++m) av[m] = a_chunk[m] < chunks ? a_voff[m] : (int)0x80000000u;
#pragma unroll
        for (int m = 0; m < C::RB; ++m) bv[m] = !C::TB || b_chunk[m] < chunks ? b_voff[m] : (int)0x80000000u;
        request<C::RA>(a_rsrc, dst + (uint32_t)wg * (C::RA * 1024u), av, a_soff);
        request<C::RB>(b_rsrc, dst + C::BM * KB + (uint32_t)wg * (C::RB * 1024u), bv, b_soff);
    };

    // ---- fragment addresses (operand lane l: row l % MF, k chunk by l / MF)
    const unsigned char* my_ring = lds + kg * (C::ST * C::STAGE);
    const int fr = lane % MF, fg = lane / MF;
    auto row_chunk = [&](int s, int h) { return ES == 2 ? s * (64 / MF) + fg : s * (128 / MF) + 2 * fg + h; };
    auto read_a = [&](const unsigned char* St, int s, int i) -> op_t {
        const int row = wm * C::WTM + i * MF + fr;
        if constexpr (ES == 2) {
            return *reinterpret_cast<const bf16x8*>(St + row * KB + swz_rows(row, row_chunk(s, 0)) * 16);
        } else {
            return join(*reinterpret_cast<const u32x4*>(St + row * KB + swz_rows(row, row_chunk(s, 0)) * 16),
                        *reinterpret_cast<const u32x4*>(St + row * KB + swz_rows(row, row_chunk(s, 1)) * 16));
        }
    };
    const int i16 = lane & 15, b16 = lane >> 4;
    auto read_b = [&](const unsigned char* St, int s, int j) -> op_t {
        const unsigned char* Bs = St + C::BM * KB;
        if constexpr (C::TB) {
            const int row = wn * C::WTN + j * MF + fr;
            if constexpr (ES == 2) {
                return *reinterpret_cast<const bf16x8*>(Bs + row * KB + swz_rows(row, row_chunk(s, 0)) * 16);
            } else {
                return join(*reinterpret_cast<const u32x4*>(Bs + row * KB + swz_rows(row, row_chunk(s, 0)) * 16),
                            *reinterpret_cast<const u32x4*>(Bs + row * KB + swz_rows(row, row_chunk(s, 1)) * 16));
            }
        } else if constexpr (ES == 2) {
            // transposing read: this lane points at 4 consecutive n of one k row; two reads give 8 k of its own n
            bf16x4 half[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int krow = MF == 32 ? 16 * s + 8 * (b16 >> 1) + 4 * h + (i16 >> 2) : 32 * s + 8 * b16 + 4 * h + (i16 >> 2);
                const int n = wn * C::WTN + j * MF + (MF == 32 ? 16 * (b16 & 1) : 0) + 4 * (i16 & 3);
                half[h] = ds_read_tr16(Bs + krow * C::B_ROW + swz_kn<C>(krow, n >> 3) * 16 + (n & 7) * 2);
            }
            return __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7);
        } else {
            u32x2 q[4];
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                const int krow = MF == 32 ? 64 * s + 32 * (b16 >> 1) + 8 * h + (i16 >> 1) : 32 * b16 + 8 * h + (i16 >> 1);
                const int n = wn * C::WTN + j * MF + (MF == 32 ? 16 * (b16 & 1) : 0) + 8 * (i16 & 1);
                q[h] = ds_read_tr8(Bs + krow * C::B_ROW + swz_kn<C>(krow, n >> 4) * 16 + (n & 15));
            }
            return join(u32x4{q[0].x, q[0].y, q[1].x, q[1].y}, u32x4{q[2].x, q[2].y, q[3].x, q[3].y});
        }
    };

    acc_t acc[C::MT][C::NT];
#pragma unroll
    for (int i = 0; i < C::MT; ++i)
#pragma unroll
        for (int j = 0; j < C::NT; ++j)
#pragma unroll
            for (int e = 0; e < MF * MF / 64; ++e) acc[i][j][e] = 0.0f;

    constexpr int REQ = C::RA + C::RB;
    struct Frags { op_t a[C::KS][C::MT], b[C::KS][C::NT]; };
    auto fragments = [&](int st, Frags& f) {
        const unsigned char* St = my_ring + st * C::STAGE;
#pragma unroll
        for (int s = 0; s < C::KS; ++s) {
#pragma unroll
            for (int i = 0; i < C::MT; ++i) f.a[s][i] = read_a(St, s, i);
#pragma unroll
            for (int j = 0; j < C::NT; ++j) f.b[s][j] = read_b(St, s, j);
        }
    };
    auto products = [&](const Frags& f) {
#pragma unroll
        for (int s = 0; s < C::KS; ++s)
#pragma unroll
            for (int i = 0; i < C::MT; ++i)
#pragma unroll
                for (int j = 0; j < C::NT; ++j) acc[i][j] = mma(f.b[s][j], f.a[s][i], acc[i][j]);
    };
    auto next = [](int st) { return st + 1 == C::ST ? 0 : st + 1; };
    // ST pieces in flight; waits leave the newer ones in flight (at the end there are fewer)
#pragma unroll
    for (int i = 0; i < C::ST; ++i)
        if (i < n_own) issue(i, i);
    // The epilogue's scales, while the first pieces are on their way: read there, each would cost its latency again (M = 1065,
    // N = 7136, K = 1024 with both vectors 15.7 us, 14.0 this way, 13.5 without any).  Products of bf16 have no vectors.
    constexpr int QPR = C::BN / 4, ROW_STEP = C::THREADS / QPR, QUADS = (C::BM + ROW_STEP - 1) / ROW_STEP;
    static_assert(C::THREADS % QPR == 0, "a lane keeps its columns");
    const int row0 = t / QPR, col = (t % QPR) * 4;
    float row_scale[QUADS];
    f32x4 col_scale{1.0f, 1.0f, 1.0f, 1.0f};
    if constexpr (ES == 1) {
#pragma unroll
        for (int i = 0; i < QUADS; ++i) row_scale[i] = 1.0f;
        if (ep.row_scale != nullptr)
#pragma unroll
            for (int i = 0; i < QUADS; ++i) row_scale[i] = ep.row_scale[min(m0 + row0 + i * ROW_STEP, M - 1)];
        if (ep.col_scale != nullptr && n0 + col < N) col_scale = *reinterpret_cast<const f32x4*>(ep.col_scale + n0 + col);
    }
    if constexpr (C::WPG == 1) {
        // the wave's own ring: no barrier.  A stage is refilled as soon as its fragments are in registers.
        Frags f;
        int st = 0;
        for (int i = 0; i < n_own; ++i) {
            if (i + C::ST <= n_own) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(REQ * (C::ST - 1)) : "memory");
            else                    wait_vmcnt0();
            fragments(st, f);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (i + C::ST < n_own) issue(i + C::ST, st);
            products(f);
            st = next(st);
        }
    } else {
        // The waves of a k-group share its stages.  Piece i + 1 is read from LDS after a barrier that every wave
        // reached with its own requests of it landed -- and with its fragments of piece i in registers, so that the
        // stage of piece i is refilled after the same barrier.  The reads run beside the products of piece i.
        // Only the last piece can be missing from a group (which keeps pace with the barriers then).
        const int n_iter = (np + C::KG - 1) / C::KG;
        Frags f0, f1;
        int st = 0;
        if (C::ST <= n_own) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(REQ * (C::ST - 1)) : "memory");
        else                wait_vmcnt0();
        __syncthreads();
        fragments(0, f0);
        int i = 0;
        auto step = [&](const Frags& cur, Frags& nxt) {
            if (i + C::ST <= n_own) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(REQ * (C::ST - 2)) : "memory");
            else                    wait_vmcnt0();
            __syncthreads();
            if (i + C::ST < n_own) issue(i + C::ST, st);
            st = next(st);
            fragments(st, nxt);
            products(cur);
            ++i;
        };
        if ((n_iter & 1) == 0 && n_iter > 0) {       // an odd number of pieces is left for the loop and the last products
            step(f0, f1);
            f0 = f1;
        }
        while (i + 1 < n_iter) {
            step(f0, f1);
            step(f1, f0);
        }
        if (i < n_own) products(f0);
    }
    // hipcc 7.2 counts 16 passes for a 32x32x64 F8F6F4 product of 8-register operands and lets the next instruction
    // read the accumulators after that many wait states; read that early the last registers of the last product came
    // out without it (found with operands of ones: exactly the last k-step was missing).
    if constexpr (ES == 1) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();

    // ---- add the k-groups in LDS and store.  Lane l of an accumulator tile holds row m = l % MF and, per register
    // group of four, 4 consecutive n.
    float* red = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int i = 0; i < C::MT; ++i)
#pragma unroll
        for (int j = 0; j < C::NT; ++j)
#pragma unroll
            for (int q = 0; q < MF * MF / 256; ++q) {
                const int row = wm * C::WTM + i * MF + fr;
                const int col = wn * C::WTN + j * MF + (MF == 32 ? 8 * q + 4 * fg : 4 * fg);
                *reinterpret_cast<f32x4*>(red + ((size_t)kg * C::BM + row) * C::RED_PITCH + col) =
                    f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
            }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < QUADS; ++i) {
        const int row = row0 + i * ROW_STEP;
        const int gm = m0 + row, gn = n0 + col;
        if (row >= C::BM || gm >= M || gn >= N) continue;
        f32x4 v = *reinterpret_cast<const f32x4*>(red + (size_t)row * C::RED_PITCH + col);
#pragma unroll
        for (int k = 1; k < C::KG; ++k) v += *reinterpret_cast<const f32x4*>(red + ((size_t)k * C::BM + row) * C::RED_PITCH + col);
        if (splits > 1) {
            *reinterpret_cast<f32x4*>(part + (((size_t)z * gridDim.y + blockIdx.y) * M + gm) * N + gn) = v;
        } else {
            if constexpr (ES == 1) v = v * (ep.scale * row_scale[i]) * col_scale;
            else                   v *= ep.scale;
            store_scaled4(ep, Cp + (size_t)blockIdx.y * stride_c * (ep.out == 1 ? 4 : ep.out == 2 ? 1 : 2), N, gm, gn, v);
        }
    }
}

// Adds the `splits` partials of every output (in the order of the K range) and applies the epilogue.
template <int ES>
__global__ __launch_bounds__(256) void gemm_tile_reduce_kernel(const float* __restrict__ part, unsigned char* __restrict__ Cp, int M, int N,
                                                               int splits, long stride_c, GemmEpilogue ep) {
    const int quads = N / 4;
    const size_t q = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= (size_t)M * quads) return;
    const int gm = (int)(q / quads), gn = (int)(q % quads) * 4;
    const size_t plane = (size_t)gridDim.y * M * N;
    const float* p = part + ((size_t)blockIdx.y * M + gm) * N + gn;
    f32x4 v = *reinterpret_cast<const f32x4*>(p);
#pragma unroll 4
    for (int z = 1; z < splits; ++z) v += *reinterpret_cast<const f32x4*>(p + z * plane);
    gt::store4(ep, Cp + (size_t)blockIdx.y * stride_c * (ep.out == 1 ? 4 : ep.out == 2 ? 1 : 2), N, gm, gn, v);
}

// ---- choice of the tile (host) ---------------------------------------------------------------------------------
// Every kernel's time is, to about 15 %, `fixed` + `piece` x (pieces a k-group walks) x (tiles the busiest of the 256 CUs
// runs): measured for bf16 and fp8 on 150 shapes with 1 <= M <= 8192 and 256 <= N, K <= 8192 and alike for both (microseconds
// on an MI355X).  The plan takes the tile and the number of K splits with the least sum; on those shapes that is 2.6 %
// slower than the best of 38 tiles tried one by one, and 3.3 times as fast as 256x256 tiles alone.
namespace gt {
// The W tiles are those with the K range shared by twice as many waves, whose rings then take a CU's whole LDS: with one
// workgroup a CU (ALONE) eight waves keep twice the pieces in flight (M = 256, N = K = 4096: fp8 10.1 -> 8.1 us, bf16 17.5 ->
// 14.6 with 64x64; M = 333 fp8 12.4 -> 10.9 with 64x128), with more the next workgroup cannot start beside the last one (M =
// 1000 28 -> 31 us).  16x16 over eight k-groups: from about 22 pieces on (M = 1, N = K = 4096 bf16 4.9 -> 4.4).
// Of 18000 drawn shapes 1935 take another plan than without them, in 10 % less time in the mean; 59 are slower by more than 2 %, the
// worst 37 % (33 x 1840 x 4928 NT bf16: 64x64W over 8 splits 8.2 us, 16x32 6.0).
enum Wide : uint8_t { NO, WIDE, ALONE };             // ALONE: WIDE, and one workgroup a CU
struct TileCost { int bm, bn, kg, mf; float fixed, piece; Wide wide = NO; };
enum Tile { T16x16, T16x16W, T16x32, T16x64, T32x32, T32x64W, T64x32, T64x32W, T64x64, T64x64W, T64x128, T64x128W, T96x64, T128x128,
            T192x128, T128x256, T256x256, TILES };
constexpr TileCost kTileCost[TILES] = {
    {16, 16, 4, 16, 2.4f, 0.19f},    {16, 16, 8, 16, 2.7f, 0.30f, WIDE},   {16, 32, 4, 16, 2.3f, 0.29f},   {16, 64, 4, 16, 2.3f, 0.43f},
    {32, 32, 4, 32, 2.4f, 0.34f},    {32, 64, 4, 32, 2.7f, 0.52f, ALONE},  {64, 32, 2, 32, 2.6f, 0.29f},   {64, 32, 4, 32, 2.7f, 0.50f, ALONE},
    {64, 64, 1, 32, 3.1f, 0.255f},   {64, 64, 2, 32, 2.9f, 0.36f, ALONE},  {64, 128, 1, 32, 3.85f, 0.34f}, {64, 128, 2, 32, 3.7f, 0.50f, ALONE},
    {96, 64, 2, 16, 3.2f, 0.71f},    {128, 128, 1, 32, 4.5f, 0.525f}, {192, 128, 1, 32, 5.5f, 0.665f}, {128, 256, 1, 32, 6.6f, 0.77f},
    {256, 256, 1, 32, 3.9f, 1.17f}};

struct Plan { int tile, splits; };

// A [K,N] B is fetched in rows of BN elements: at least 64 bytes of each.
inline bool tile_takes(int tile, int es, bool tb) { return tb || kTileCost[tile].bn * es >= 64; }

// What a caller allows.  The order in which K is summed depends on the MFMA shape, the k-groups and the splits, not on the rest of the
// tile.  BATCH: the order that the same product has as an entry of a batch, so that both give the same bits; a batch picks its tile
// among those.  The W tiles are not for it (bf16; there are no batches of e4m3): a large batch would be left with one small tile of
// their order.  ANY: without scratch for partials.  SPLIT: with.
enum Sums : uint8_t { BATCH, ANY, SPLIT };

inline double tile_cost(int tile, int splits, int M, int N, int K, int es, bool tb, int batch, Sums sums) {
    const TileCost& t = kTileCost[tile];
    const int64_t pieces = ((int64_t)K * es + KB - 1) / KB, per_split = (pieces + splits - 1) / splits;
    const int64_t tiles = (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * splits * batch;
    if (t.wide == ALONE && tiles > 256) return 1e30;
    // Rows that do not start on cache lines, or are half a line: every piece of one touches two.  A CU's requests are what bounds an
    // ALONE tile (64x64W, 44 pieces of 126 x 6992 x 5544 bf16: 0.57 us each for 0.36) and 16x16W with more than 16 rows on all CUs
    // (173 x 352 x 4456 NT bf16 5.2 us with 16x16, 5.9 with 16x16W), the others wait as much for other things (1.16 x).
    const bool half = !tb && t.bn * es < KB;
    const bool lines = (int64_t)K * es % KB == 0 && (tb || ((int64_t)N * es % KB == 0 && !half));
    double piece = !lines && (t.wide == ALONE || (t.wide == WIDE && tiles > 200 && M > t.bm)) ? 1.4 * t.piece : t.piece;
    // The ring of 96x64 takes a CU's whole LDS too: its 0.71 us hold that every further round starts anew.  2719 x 448 x 1280 NN
    // bf16, one round of 10 pieces a k-group, 8.2 us (64x128W 8.7).  Not where its order of sums would bind a batch, which has no
    // other tile of that order.
    if (tile == T96x64 && es == 2 && sums != BATCH && splits == 1 && tiles <= 256 && pieces <= 64) piece = 0.53;
    double us = t.fixed + piece * ((per_split + t.kg - 1) / t.kg) * ((tiles + 255) / 256);
    // Half lines of a long [K,N] B, where K can be split instead (the other tiles that take it whole are slower still): 549 x 736 x
    // 7936 e4m3 17.9 us with 32x64W, 13.3 with 64x128 over 4 splits.
    if (t.wide == ALONE && half && sums == SPLIT && per_split > 40) us += 0.1 * (per_split - 40);
    // the second kernel, and f32 partials written and read at 5 TB/s
    if (splits > 1) us += 2.6 + (double)M * N * batch * 8.0 * splits / 5.0e6;
    // no tile is faster than memory; among those that reach it the one with the least to do still wins
    const double memory = 2.3 + batch * ((double)es * K * ((double)M + N) + 2.0 * M * N) / 6.0e6;
    return (us > memory ? us : memory) + 0.05 * us;
}

inline Plan make_plan(int M, int N, int K, int es, bool tb, int batch, Sums sums) {
    if (batch > 1) sums = BATCH;
    Plan best{T256x256, 1};
    double least = tile_cost(T256x256, 1, M, N, K, es, tb, 1, sums);
    const int64_t pieces = ((int64_t)K * es + KB - 1) / KB;
    for (int tile = 0; tile < T256x256; ++tile) {
        if (!tile_takes(tile, es, tb) || (kTileCost[tile].wide && es == 2 && sums == BATCH)) continue;
        for (int splits = 1; splits <= 8; ++splits) {
            if (splits > 1 && (sums != SPLIT || pieces < 4 * splits)) break;
            const double us = tile_cost(tile, splits, M, N, K, es, tb, 1, sums);
            if (us < least) { least = us; best = {tile, splits}; }
        }
    }
    if (batch > 1) {
        const TileCost order = kTileCost[best.tile];
        least = tile_cost(best.tile, 1, M, N, K, es, tb, batch, BATCH);
        for (int tile = 0; tile < TILES; ++tile) {
            if (!tile_takes(tile, es, tb) || kTileCost[tile].wide || kTileCost[tile].kg != order.kg || kTileCost[tile].mf != order.mf) continue;
            const double us = tile_cost(tile, 1, M, N, K, es, tb, batch, BATCH);
            if (us < least) { least = us; best.tile = tile; }
        }
    }
    // as many splits as there are whole ranges of ceil(pieces / splits)
    const int64_t per_split = (pieces + best.splits - 1) / best.splits;
    best.splits = (int)((pieces + per_split - 1) / per_split);
    return best;
}

inline size_t scratch_bytes(const Plan& p, int M, int N, int batch) {
    return p.splits > 1 ? (size_t)p.splits * batch * M * N * sizeof(float) : 0;
}

// make_plan costs about a microsecond of host time; a program repeats few shapes, so each thread keeps its last plans.
inline Plan plan(int M, int N, int K, int es, bool tb, int batch, Sums sums) {
    struct Entry { int M, N, K, batch, kind; Plan plan; };
    static thread_local Entry kept[64];
    const int kind = 1 + (es * 2 + tb) * 3 + sums;                   // 0 = an unused entry
    const uint32_t h = ((uint32_t)M * 0x9e3779b1u ^ (uint32_t)N * 0x85ebca6bu ^ (uint32_t)K * 0xc2b2ae35u ^ (uint32_t)batch * 0x27d4eb2fu ^ (uint32_t)kind) * 0x9e3779b1u;
    Entry& e = kept[h >> 26];
    if (e.kind != kind || e.M != M || e.N != N || e.K != K || e.batch != batch)
        e = {M, N, K, batch, kind, make_plan(M, N, K, es, tb, batch, sums)};
    return e.plan;
}
inline Plan plan_within(int M, int N, int K, int es, bool tb, int batch, const void* workspace, size_t workspace_bytes) {
    if (workspace == nullptr) return plan(M, N, K, es, tb, batch, BATCH);
    const Plan p = plan(M, N, K, es, tb, batch, SPLIT);
    return scratch_bytes(p, M, N, batch) <= workspace_bytes ? p : plan(M, N, K, es, tb, batch, ANY);
}

template <class C>
int launch(const void* a, const void* b, void* c, int M, int N, int K, int splits, float* part, int batch, int64_t stride_a,
           int64_t stride_b, int64_t stride_c, const GemmEpilogue& ep, hipStream_t stream) {
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_tile_kernel<C>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
    if (attr != hipSuccess) return -1;
    const int tiles_m = (M + C::BM - 1) / C::BM, tiles_n = (N + C::BN - 1) / C::BN;
    const int64_t wgs = (int64_t)tiles_m * tiles_n * splits;
    if (wgs > INT_MAX) return -1;
    // the 8 XCDs' shares of the tiles: about as high as wide
    int group_m = (int)lround(sqrt((double)tiles_m * tiles_n / 8 * C::BN / C::BM));
    group_m = group_m < 1 ? 1 : group_m > tiles_m ? tiles_m : group_m;
    const int pieces = (int)(((int64_t)K * C::ES + KB - 1) / KB), per_split = (pieces + splits - 1) / splits;
    launch_kernel((gemm_tile_kernel<C>), dim3((unsigned)wgs, (unsigned)batch), dim3(C::THREADS), C::LDS, stream,
                       static_cast<const unsigned char*>(a), static_cast<const unsigned char*>(b), static_cast<unsigned char*>(c), part, M, N,
                       K, tiles_m, tiles_n, group_m, splits, pieces, per_split, (long)stride_a, (long)stride_b, (long)stride_c, ep);
    if (hipGetLastError() != hipSuccess) return -1;
    if (splits > 1) {
        launch_kernel(gemm_tile_reduce_kernel<C::ES>, dim3((unsigned)(((size_t)M * (N / 4) + 255) / 256), (unsigned)batch), dim3(256), 0,
                           stream, part, static_cast<unsigned char*>(c), M, N, splits, (long)stride_c, ep);
        if (hipGetLastError() != hipSuccess) return -1;
    }
    return 0;
}

// p.tile != T256x256
template <int ES, bool TB>
int launch_plan(const Plan& p, const void* a, const void* b, void* c, int M, int N, int K, float* part, int batch, int64_t stride_a,
                int64_t stride_b, int64_t stride_c, const GemmEpilogue& ep, hipStream_t stream) {
#define TYR_TILE(NAME, BM, BN, WTM, WTN, KG, ST)                                                                              \
    case NAME:                                                                                                                \
        if constexpr (TB || BN * ES >= 64)                                                                                    \
            return launch<Cfg<ES, TB, BM, BN, WTM, WTN, KG, ST>>(a, b, c, M, N, K, p.splits, part, batch, stride_a, stride_b, \
                                                                 stride_c, ep, stream);                                       \
        return -1;
    switch (p.tile) {
        TYR_TILE(T16x16, 16, 16, 16, 16, 4, 4)
        TYR_TILE(T16x16W, 16, 16, 16, 16, 8, 2)
        TYR_TILE(T16x32, 16, 32, 16, 32, 4, 3)
        TYR_TILE(T16x64, 16, 64, 16, 64, 4, 2)
        TYR_TILE(T32x32, 32, 32, 32, 32, 4, 2)
        TYR_TILE(T32x64W, 32, 64, 32, 32, 4, 3)
        TYR_TILE(T64x32, 64, 32, 32, 32, 2, 3)
        TYR_TILE(T64x32W, 64, 32, 32, 32, 4, 3)
        TYR_TILE(T64x64, 64, 64, 32, 32, 1, 5)
        TYR_TILE(T64x64W, 64, 64, 32, 32, 2, 3)
        TYR_TILE(T64x128, 64, 128, 64, 32, 1, 3)
        TYR_TILE(T64x128W, 64, 128, 64, 32, 2, 3)
        TYR_TILE(T96x64, 96, 64, 48, 32, 2, 4)
        TYR_TILE(T128x128, 128, 128, 64, 32, 1, 5)
        TYR_TILE(T192x128, 192, 128, 96, 32, 1, 4)
        TYR_TILE(T128x256, 128, 256, 64, 64, 1, 3)
        default: return -1;
    }
#undef TYR_TILE
}

// Offsets are 32 bits wide: a tile's rows of A (and of a [N,K] B) stay below 2 GiB, a [K,N] B below 4 GiB.
inline bool offsets_fit(int N, int K, int es, bool tb) {
    return (size_t)256 * K * es < ((size_t)1 << 31) && (tb || (size_t)K * N * es < ((size_t)1 << 32) - 4096);
}
}  // namespace gt

}  // namespace tyr
