// Flash-attention backward for gfx950 (bf16 in, f32 accumulation, bf16 dQ / dK / dV).
//
// Arithmetic contract of the reference (Tyr/GPU/Kernels/MhaH100.lean):
//   :197-232  backward prep      delta[i] = sum_d dO[i,d] * O[i,d]
//   :234-344  backward           S = Q K^T * scale ; P = exp(S - lse) ; dP = dO V^T ;
//                                dS = P o (dP - delta) ; dV += bf16(P)^T dO ;
//                                dK += bf16(dS)^T Q * scale ; dQ += bf16(dS) K * scale
// (expected values in the reference's runner come from autograd of scaled_dot_product_attention,
// Examples/GPU/RunMhaH100.lean:56-64).  exp is evaluated as exp2 with log2(e) folded into the
// scale and into the saved log-sum-exp.  causal: key j visible to query i iff j <= i.
//
// Two kernels (one launch where they leave CUs idle), no atomics, every output written once (results are deterministic):
//
//  1. flash_attn_bwd_dq_kernel: one workgroup = 128 query rows (4 waves x 32 rows), keys/values
//     stream through LDS in tiles of 64 rows exactly as in the forward kernel.  Products are
//     computed transposed so that every lane owns one query column:
//        S^T  (64 kv x 32 q) = K_tile x Q^T       dP^T (64 kv x 32 q) = V_tile x dO^T
//        dQ^T (D x 32 q)    += K_tile^T x dS^T
//     so lse and delta are per-lane scalars and dS^T is already in the register slots the third
//     product wants as its column operand.  The prologue also computes delta (each wave holds its
//     dO rows and reads its O rows once) and writes (lse * log2 e, delta) pairs to the workspace
//     for the second kernel; rows of the padding up to a multiple of 128 get (+inf, 0), which
//     makes their probabilities exactly zero.
//
//  2. flash_attn_bwd_dkv_kernel: one workgroup = 128 key rows (4 waves x 32 rows, K and V
//     fragments of those rows live in registers), queries / dO stream through LDS in tiles of 64
//     rows, four stages deep.  Every lane owns one key column:
//        S  (32 q x 32 kv) = Q_tile x K_w^T        dP (32 q x 32 kv) = dO_tile x V_w^T
//        dV^T (D x 32 kv) += dO_tile^T x P         dK^T (D x 32 kv) += Q_tile^T x dS
//     with lse / delta of the 16 query rows a lane holds read from the staged pairs.  Launches of many key tiles take
//     flash_attn_bwd_dkv_wide_kernel, 256 keys a workgroup; small ones bwd_dkv_half, 64 keys.
//
// Both recompute S (7 matrix products for an algorithm that needs 5): the price of writing dQ
// without a float atomic accumulation buffer and a conversion pass.
//
// Where that is faster (launch_us), and dS fits, the 5 products run: flash_attn_bwd_stats_kernel makes the pairs, dK/dV goes first and leaves
// its bf16 dS in the workspace, and flash_attn_bwd_dq_product_kernel adds dQ = dS K from there.  Same operands and roundings.
//
// LDS tiles are row-major with 16-byte chunks XOR-swizzled by a function of the row that is
// conflict-free both for row fragments (16-byte reads, lane = row) and for transposed fragments
// (ds_read_b64_tr_b16 over 4 rows x 64 bytes per lane-group pair).
#include <limits.h>

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"

namespace tyr {

namespace fab {
constexpr int THREADS = 256;
constexpr float LOG2E = 1.4426950408889634f;

// chunk index within a row -> stored chunk index.  The mask is a bijection of (row mod 16) [of
// ((row / 2) mod 8) for 128-byte rows], so 16 consecutive rows put one logical chunk on 16
// different bank groups; its upper bits follow row mod 4, which spreads the 4 rows a lane group
// of the transposing read touches over the 4 64-byte quarters of the bank space.
template <int D> __device__ __forceinline__ int swz(int row, int c) {
    return D == 128 ? (c ^ (((row & 3) << 2) | ((row >> 2) & 3)))
                    : (c ^ ((((row >> 1) & 1) << 2) | ((row >> 2) & 3)));
}

template <int D>
struct CfgQ {                                       // dQ kernel
    static constexpr int BM = 128, BN = 64;
    static constexpr int ROW = D * 2, KCH = D / 8;
    static constexpr int TILE = BN * ROW;
    static constexpr int V_BASE = 2 * TILE;         // K stage 0, K stage 1, V stage 0, V stage 1
    static constexpr int LDS = 4 * TILE;
    static constexpr int PT = BN * KCH / THREADS;   // 16-byte chunks per thread per tile
    static constexpr int KSTEPS = D / 16, DT = D / 32;
};

template <int D>
struct CfgK {                                       // dK / dV kernel
    static constexpr int BNK = 128, BQ = 64, NST = 4;   // NST must stay a power of two
    static constexpr int ROW = D * 2, KCH = D / 8;
    static constexpr int TILE = BQ * ROW;
    static constexpr int STAT = 1024;               // 64 (lse2, delta) pairs + slack of one load
    static constexpr int STAGE = 2 * TILE + STAT;   // Q tile, dO tile, pairs
    static constexpr int LDS = NST * STAGE;
    static constexpr int PT = BQ * KCH / THREADS;
    static constexpr int KSTEPS = D / 16, DT = D / 32;
    static constexpr int LOADS_PER_TILE = 2 * PT + 1;
};

__device__ __forceinline__ float dot8_bf16(u32x4 a, u32x4 b) {
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) s += bf16_lo(a[i]) * bf16_lo(b[i]) + bf16_hi(a[i]) * bf16_hi(b[i]);
    return s;
}

// What the dK / dV workgroups need of a query row: (lse * log2 e, delta), or with fours = 3, for the wide kernel, by groups of four rows
// four lse * log2 e and four -delta (16 bytes each: what a lane's scores need; its dP starts from -delta).  One pair of stores for
// both, and nothing for the compiler to keep across the passes of a workgroup (row & 3 is the same in each): as a branch the dQ
// kernels held two registers more, and at 170 for 168 two waves of <64, causal, Keys, SPLIT> share a SIMD for three.
__device__ __forceinline__ void store_stats(float2* head, int row, float lse2, float delta, int fours) {
    asm volatile("" : "+v"(row));
    float* at = reinterpret_cast<float*>(head) + (2 * row - (row & fours));
    at[0] = lse2;
    at[1 + fours] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, delta) ^ ((uint32_t)fours << 31));
}

// One wave's 32 columns x D rows accumulator (lane = column l%32, register e of tile dt <-> row
// 32 dt + 8(e/4) + 4(l/32) + e%4), scaled, written as bf16 rows of length D: out row = column.
// Goes through a private LDS scratch so the global stores are 16 bytes per lane along rows.
template <int D>
__device__ __forceinline__ void store_transposed_bf16(const f32x16 (&acc)[D / 32], float mul, unsigned char* scratch,
                                                      uint16_t* out_rows, int rows_valid, int lane) {
    constexpr int SROW = D * 2 + 16;
    const int r = lane & 31, g = lane >> 5;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt) {
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            u32x2 v;
            v.x = pack_bf16(acc[dt][4 * q4 + 0] * mul, acc[dt][4 * q4 + 1] * mul);
            v.y = pack_bf16(acc[dt][4 * q4 + 2] * mul, acc[dt][4 * q4 + 3] * mul);
            *reinterpret_cast<u32x2*>(scratch + r * SROW + (dt * 32 + q4 * 8 + g * 4) * 2) = v;
        }
    }
    constexpr int CH = D / 8;
    constexpr int RPI = 64 / CH;
#pragma unroll
    for (int k = 0; k < 32 / RPI; ++k) {
        const int row = lane / CH + RPI * k;
        const u32x4 v = *reinterpret_cast<const u32x4*>(scratch + row * SROW + (lane % CH) * 16);
        if (row < rows_valid) st_global_16(out_rows + (size_t)row * D + (lane % CH) * 8, v);
    }
}
}  // namespace fab

// ------------------------------------------------------------------------------------------
// dQ (and the (lse2, delta) pairs)
// MASK as in the forward kernel;
// G = query heads per kv head.  SPLIT: 64 query rows per workgroup, the two 32-key sub-tiles of a tile on two waves whose
// dQ are added through LDS at the end (same use as in the forward kernel: launches with few tiles).  Not causal at D = 128, 41 to
// 52 registers are too many for two waves a SIMD (168 to 212 bytes a lane in scratch memory; causal none).
template <int D, bool CAUSAL, AttnMask MASK, bool SPLIT>
__device__ __forceinline__ void bwd_dq(int block,
    const uint16_t* __restrict__ Q, const uint16_t* __restrict__ Kp, const uint16_t* __restrict__ Vp,
    const uint16_t* __restrict__ O, const uint16_t* __restrict__ dO, const float* __restrict__ LSE,
    uint16_t* __restrict__ dQ, float2* __restrict__ stats, int BH, int N, int ntq, int npad, float scale,
    float scale_log2, int Hq, int G, int window, const int* __restrict__ kv_lens,
    const uint8_t* __restrict__ key_mask, int pair, int single, int fours) {
    using namespace fab;
    using C = CfgQ<D>;
    constexpr bool LIMITS = MASK == AttnMask::Limits, KEYS = MASK == AttnMask::Keys;
    constexpr int TBM = SPLIT ? 64 : C::BM;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

    const int t = threadIdx.x;
    const int lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int r = lane & 31, g = lane >> 5;
    const int wr = SPLIT ? w & 1 : w;            // which 32 rows of the tile
    const int T0 = SPLIT ? w >> 1 : 0;           // SPLIT: the one sub-tile of this wave

    // With `pair` (causal) a workgroup handles query tile ntq-1-tr and then tile tr.
    int bh, tr, kvbh;
    AttnOrder{BH, Hq, G, pair ? (ntq + 1) / 2 : ntq, single}.decode(block, bh, tr, kvbh);
    const int npass = (pair && ntq - 1 - tr != tr) ? 2 : 1;
    for (int pass = 0; pass < npass; ++pass) {
    const int qt = CAUSAL ? (pass == 0 ? ntq - 1 - tr : tr) : tr;
    const int q0 = qt * TBM;
    const int qw0 = q0 + wr * 32;
    const size_t head_off = (size_t)bh * N * D;
    const uint16_t* Kh = Kp + (size_t)kvbh * N * D;
    const uint16_t* Vh = Vp + (size_t)kvbh * N * D;
    const int Nk = (LIMITS && kv_lens != nullptr) ? max(0, min(N, kv_lens[bh / Hq])) : N;
    const uint8_t* km = KEYS ? key_mask + (size_t)(bh / Hq) * N : nullptr;
    const int kv_end = CAUSAL ? min(Nk, q0 + TBM) : Nk;
    const int nkv_abs = max(1, (kv_end + C::BN - 1) / C::BN);   // a sequence without keys still walks one (fully masked) tile
    int jbase = (LIMITS && window > 0) ? min(max(0, q0 - window + 1) / C::BN, nkv_abs - 1) : 0;
    int nkv = nkv_abs - jbase;                   // tiles are numbered from jbase below
    const int qpos = qw0 + r;

    // ---- this wave's Q^T and dO^T fragments (lane = query row, columns 16i + 8g + [0,8)),
    //      delta = dO . O and lse in log2 units
    bf16x8 qf[C::KSTEPS], dof[C::KSTEPS];
    float delta, lse2;
    {
        const int qrow = min(qpos, N - 1);
        const size_t off = head_off + (size_t)qrow * D + g * 8;
        float part = 0.0f;
#pragma unroll
        for (int i = 0; i < C::KSTEPS; ++i) {
            qf[i] = __builtin_bit_cast(bf16x8, ld_global_16(Q + off + i * 16));
            const u32x4 dv = ld_global_16(dO + off + i * 16);
            const u32x4 ov = ld_global_16(O + off + i * 16);
            dof[i] = __builtin_bit_cast(bf16x8, dv);
            part += dot8_bf16(dv, ov);
        }
        delta = part + xor32(part);
        lse2 = LSE[(size_t)bh * N + qrow] * LOG2E;
        if (MASK != AttnMask::None && lse2 == -INFINITY) lse2 = INFINITY;      // a row that saw no key: every probability is 0
        if (stats != nullptr && g == 0 && T0 == 0) {
            store_stats(stats + (size_t)bh * npad, qpos, qpos < N ? lse2 : INFINITY, qpos < N ? delta : 0.0f, fours);
        }
    }

    // ---- K / V tile loaders (global memory straight into LDS, swizzle applied on the global side)
    const uint32_t head_bytes = (uint32_t)N * D * 2u;
    const u32x4 k_rsrc = make_raw_rsrc(Kh, head_bytes);
    const u32x4 v_rsrc = make_raw_rsrc(Vh, head_bytes);
    constexpr int ROWS_PER_INST = 1024 / C::ROW;
    int g_voff[C::PT];
#pragma unroll
    for (int m = 0; m < C::PT; ++m) {
        const int row = (w * C::PT + m) * ROWS_PER_INST + lane / C::KCH;
        g_voff[m] = row * C::ROW + swz<D>(row, lane % C::KCH) * 16 - 1024 * m;   // request m carries 1024 m as its immediate offset
    }
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
    const uint32_t wave_dst = __builtin_amdgcn_readfirstlane(lds_base + (uint32_t)w * C::PT * 1024u);
    auto issue_kv = [&](int stage, int j0) {
        const uint32_t dst = wave_dst + (uint32_t)stage * C::TILE;
        load_global_to_lds_16xN<C::PT>(k_rsrc, dst, g_voff, j0 * C::ROW);
        load_global_to_lds_16xN<C::PT>(v_rsrc, dst + C::V_BASE, g_voff, j0 * C::ROW);
    };

    // row fragment (sub-tile T, k-step i): row 32T + r, chunk 2i + g
    int row_off[C::KSTEPS];
#pragma unroll
    for (int i = 0; i < C::KSTEPS; ++i) row_off[i] = r * C::ROW + swz<D>(r, 2 * i + g) * 16;
    // transposed fragment (d tile dt; kv rows 16c + 8h + 4g + [0,4)): as a source lane of the
    // transposing read this lane points at row 4(b/2) + (lane%16)/4 (+8 for the second read),
    // 8 bytes at d = 32dt + 16(b&1) + 4(lane%4), b = lane/16.
    int tr_lo[C::DT], tr_hi[C::DT];
    {
        const int i16 = lane & 15, b16 = lane >> 4;
        const int row = 4 * (b16 >> 1) + (i16 >> 2);
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt) {
            const int dcol = 32 * dt + 16 * (b16 & 1) + 4 * (i16 & 3);
            tr_lo[dt] = row * C::ROW + swz<D>(row, dcol >> 3) * 16 + (dcol & 7) * 2;
            tr_hi[dt] = (row + 8) * C::ROW + swz<D>(row + 8, dcol >> 3) * 16 + (dcol & 7) * 2;
        }
    }

    f32x16 dq[C::DT];
#pragma unroll
    for (int i = 0; i < C::DT; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) dq[i][e] = 0.0f;

    issue_kv(0, jbase * C::BN);
    uint64_t next_hidden = 0;                    // KEYS: bit r set = kv row r of the next step's tile is hidden
    if constexpr (KEYS) {                        // tiles before the first and after the last visible key are not walked
        const TileSpan span = visible_tiles(km, kv_end, lane);
        const int end = max(1, span.last);
        jbase = min(span.first, end - 1);
        nkv = end - jbase;
        if (jbase > 0) {
            wait_vmcnt0();
            issue_kv(0, jbase * C::BN);
        }
        next_hidden = __builtin_amdgcn_ballot_w64(km[min(jbase * C::BN + lane, N - 1)] == 0);
    }
    const int nkv_w = CAUSAL ? min(nkv, (qw0 + 31) / C::BN + 1 - jbase) : nkv;

#pragma unroll
    for (int i = 0; i < C::KSTEPS; ++i) { pin_registers(qf[i]); pin_registers(dof[i]); }
    wait_vmcnt0();
    __syncthreads();

    for (int j = 0; j < nkv; ++j) {
        const int j0 = (jbase + j) * C::BN;
        // the tile's 64 key-mask bytes as one word (bit r set: kv row j0 + r is hidden): one byte per lane and a ballot,
        // read one step ahead; a tile without hidden rows skips the masking
        const uint64_t tile_hidden = next_hidden;
        uint32_t mask_byte = 1;
        if (KEYS && j + 1 < nkv) mask_byte = km[min(j0 + C::BN + lane, N - 1)];
        if (j + 1 < nkv) issue_kv((j + 1) & 1, j0 + C::BN);
        if (j < nkv_w) {
            const unsigned char* Kt = lds + (j & 1) * C::TILE + (SPLIT ? T0 * 32 * C::ROW : 0);
            const unsigned char* Vt = Kt + C::V_BASE;
            // The two 32-row sub-tiles of the tile are taken one after the other (scores, probabilities, dQ
            // products): only one sub-tile's scores are live, which leaves the registers the fragment read-ahead
            // needs; the other wave of the SIMD has matrix work while this one does its exponentials.
            f32x16 s[2], dp[2];
            bf16x8 dsf[4];
            const bool need_mask = (CAUSAL && (j0 + C::BN - 1 > qw0)) || (j0 + C::BN > Nk) ||
                                   (LIMITS && window > 0 && j0 < qw0 + 32 - window) || (KEYS && tile_hidden != 0);
            // Fragments are read one k-step ahead of the products that take them, also across the phases of a tile (the
            // first fragments of a phase are requested under the last products of the phase before it), and the
            // scheduling barriers keep that order: left to itself the compiler, at its register limit, puts every read
            // right in front of its product and the wave waits out the LDS latency 48 times per tile.
            bf16x8 ka[2], va[2];                 // K / V row fragments of the scores phase
            bf16x4 lo[2], hi[2];                 // transposed K fragments of the dQ phase
            auto read_rows = [&](int T, int i, int slot) {
                ka[slot] = *reinterpret_cast<const bf16x8*>(Kt + row_off[i] + T * 32 * C::ROW);
                va[slot] = *reinterpret_cast<const bf16x8*>(Vt + row_off[i] + T * 32 * C::ROW);
            };
            auto read_transposed = [&](int T, int n, int slot) {      // n = (c - 2T) * DT + dt
                const int c = 2 * T + n / C::DT, dt = n % C::DT;
                lo[slot] = ds_read_tr16(Kt + tr_lo[dt] + c * 16 * C::ROW);
                hi[slot] = ds_read_tr16(Kt + tr_hi[dt] + c * 16 * C::ROW);
            };
            auto scores = [&](int T) {           // expects the fragments of k-step 0 in slot 0
#pragma unroll
                for (int e = 0; e < 16; ++e) { s[T][e] = 0.0f; dp[T][e] = 0.0f; }
#pragma unroll
                for (int i = 0; i < C::KSTEPS; ++i) {
                    if (i + 1 < C::KSTEPS) read_rows(T, i + 1, (i + 1) & 1);
                    else read_transposed(T, 0, 0);               // first fragment of this sub-tile's dQ phase
                    __builtin_amdgcn_sched_barrier(0);
                    s[T] = mfma_32x32x16_bf16(ka[i & 1], qf[i], s[T]);
                    dp[T] = mfma_32x32x16_bf16(va[i & 1], dof[i], dp[T]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            // mask (diagonal tiles, ragged tail), then dS^T = P^T o (dP^T - delta) packed into column-operand
            // slots (group c = 2T + sh holds registers 8sh .. 8sh+7 of sub-tile T).  Register e of sub-tile T
            // is kv row j0 + 32T + 8(e/4) + 4g + e%4.
            auto probabilities = [&](int T) {
                if (need_mask) {
                    const int lim = CAUSAL ? min(qpos, Nk - 1) : Nk - 1;
                    const int low = (LIMITS && window > 0) ? qpos - window + 1 : INT_MIN;
                    const int base = j0 + 32 * T0 + 4 * g;
                    const uint64_t hidden = tile_hidden >> (4 * g + 32 * (T0 + T));      // shifted to this lane's rows
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int kv = base + 32 * T + 8 * (e >> 2) + (e & 3);
                        const bool off = kv > lim || (LIMITS && kv < low) || ((hidden >> (8 * (e >> 2) + (e & 3))) & 1u);
                        s[T][e] = off ? -INFINITY : s[T][e];
                    }
                }
#pragma unroll
                for (int sh = 0; sh < 2; ++sh) {
                    u32x4 pk;
#pragma unroll
                    for (int jj = 0; jj < 4; ++jj) {
                        const int e = 8 * sh + 2 * jj;
                        const float p0 = fast_exp2(fmaf(s[T][e], scale_log2, -lse2));
                        const float p1 = fast_exp2(fmaf(s[T][e + 1], scale_log2, -lse2));
                        pk[jj] = pack_bf16(p0 * (dp[T][e] - delta), p1 * (dp[T][e + 1] - delta));
                    }
                    dsf[2 * T + sh] = __builtin_bit_cast(bf16x8, pk);
                }
            };
            // dQ^T += K^T dS^T for the two 16-row groups of sub-tile T
            auto accumulate = [&](int T) {       // expects the transposed fragment 0 in slot 0
#pragma unroll
                for (int n = 0; n < 2 * C::DT; ++n) {
                    const int c = 2 * T + n / C::DT, dt = n % C::DT;
                    if (n + 1 < 2 * C::DT) read_transposed(T, n + 1, (n + 1) & 1);
                    else if (T == 0 && !SPLIT) read_rows(1, 0, 0);   // first fragments of the second sub-tile's scores
                    __builtin_amdgcn_sched_barrier(0);
                    const bf16x8 kt = __builtin_shufflevector(lo[n & 1], hi[n & 1], 0, 1, 2, 3, 4, 5, 6, 7);
                    dq[dt] = mfma_32x32x16_bf16(kt, dsf[c], dq[dt]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            if constexpr (SPLIT) {
                // one sub-tile per wave: register arrays are indexed as sub-tile 0, addresses and masks are of sub-tile T0
                read_rows(0, 0, 0);
                scores(0);
                probabilities(0);
                accumulate(0);
            } else {
                read_rows(0, 0, 0);
                scores(0);
                probabilities(0);
                accumulate(0);
                scores(1);
                probabilities(1);
                accumulate(1);
            }
        }
        wait_vmcnt0();
        if constexpr (KEYS) next_hidden = __builtin_amdgcn_ballot_w64(mask_byte == 0);
        __syncthreads();
    }

    if constexpr (SPLIT) {
        f32x4* other = reinterpret_cast<f32x4*>(lds) + wr * (C::DT * 4 * 64) + lane;
        if (w >= 2) {
#pragma unroll
            for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4)
                    other[(dt * 4 + q4) * 64] = f32x4{dq[dt][4 * q4], dq[dt][4 * q4 + 1], dq[dt][4 * q4 + 2], dq[dt][4 * q4 + 3]};
        }
        __syncthreads();
        if (w < 2) {
#pragma unroll
            for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) {
                    const f32x4 o = other[(dt * 4 + q4) * 64];
#pragma unroll
                    for (int x = 0; x < 4; ++x) dq[dt][4 * q4 + x] += o[x];
                }
            store_transposed_bf16<D>(dq, scale, lds + C::LDS / 2 + w * (32 * (D * 2 + 16)), dQ + head_off + (size_t)qw0 * D,
                                     N - qw0, lane);
        }
    } else {
        store_transposed_bf16<D>(dq, scale, lds + w * (32 * (D * 2 + 16)), dQ + head_off + (size_t)qw0 * D,
                                 N - qw0, lane);
    }
    __syncthreads();                             // the scratch is read; the stages may be refilled
    }
}

template <int D, bool CAUSAL, AttnMask MASK, bool SPLIT>
__global__ __launch_bounds__(fab::THREADS, 2) void flash_attn_bwd_dq_kernel(
    const uint16_t* __restrict__ Q, const uint16_t* __restrict__ Kp, const uint16_t* __restrict__ Vp,
    const uint16_t* __restrict__ O, const uint16_t* __restrict__ dO, const float* __restrict__ LSE,
    uint16_t* __restrict__ dQ, float2* __restrict__ stats, int BH, int N, int ntq, int npad, float scale,
    float scale_log2, int Hq, int G, int window, const int* __restrict__ kv_lens,
    const uint8_t* __restrict__ key_mask, int pair, int single, int fours) {
    bwd_dq<D, CAUSAL, MASK, SPLIT>(blockIdx.x, Q, Kp, Vp, O, dO, LSE, dQ, stats, BH, N, ntq, npad, scale, scale_log2, Hq, G, window,
                                   kv_lens, key_mask, pair, single, fours);
}

// ------------------------------------------------------------------------------------------
// dK, dV
// BHkv = batch * kv heads; the G query heads of a kv head are walked one after the other and
// accumulate into the same dK / dV (the gradient of repeat_interleave).  A lane owns one
// key, so lengths and key masks (Keys) need no instructions in the steps: what a hidden key's lane summed is set to zero at
// the end, and a block of 128 hidden keys walks no query (padded batch of 8, 2000 rows, whole backward: 933 -> 428 us with a
// key mask, 747 -> 558 with lengths).  Limits is a window, with or without lengths: its steps carry mask instructions.
// Where (key tile, kv head) pairs are too few or too unequal for the device (causal: the first key tile meets every query
// tile, the last one two; all times G), the steps of a key tile -- its 64-row query tiles, head after head -- are cut
// into equal parts of at most `chunk` for as many workgroups, which leave f32 partial sums that flash_attn_bwd_sum_kernel adds.
namespace fab {
struct Parts {
    int G, nq, causal, window, chunk;                // chunk = 0: one part per key tile
    int keys;                                        // of a key tile: 128, or 256 (flash_attn_bwd_dkv_wide_kernel, chunk = 0)
    // 64-row query tiles that see key tile kt: [first(kt), last(kt))
    __host__ __device__ int first(int kt) const { return causal ? keys / 64 * kt : 0; }
    __host__ __device__ int last(int kt) const {
        if (window <= 0) return nq;                  // the last query that sees a key of the tile is keys (kt + 1) - 1 + window - 1
        const int64_t e = ((int64_t)keys * kt + keys - 2 + window) / 64 + 1;
        return e < nq ? (int)e : nq;
    }
    __host__ __device__ int steps(int kt) const { return G * (last(kt) - first(kt)); }
    __host__ __device__ int parts(int kt) const { return chunk == 0 ? 1 : (steps(kt) + chunk - 1) / chunk; }
    __host__ __device__ int part_steps(int kt) const { const int n = parts(kt); return (steps(kt) + n - 1) / n; }
    // Whole key tiles: the head (of those of an XCD, or of all) and the key tile of workgroup `slot`.  An XCD deals its workgroups
    // to its four shader engines in turn, in order: one whose engine has no free CU holds up all behind it.  Causal tiles are of
    // unequal length (the first meets every query tile, the last one two), so neighbours in the order are the same tile of eight
    // heads.  Head after head instead, CUs stood idle for 5 to 25 %
    // of the launch: dK/dV of B16 H16 N4096 2367 us, 2232 in this order, of B32 H32 N512 362 and 273, at D = 64 of B16 H32 N1024 324 and 266.
    // Equal tiles go head after head: their Q / dO then share the L2.
    __host__ __device__ int order(int slot, int heads, bool xcds, int tiles, int& kt) const {
        const int unit = causal && window <= 0 ? (xcds ? 8 : 32) : 1;
        const int first = slot / (unit * tiles) * unit, n = heads - first < unit ? heads - first : unit;
        const int at = slot - first * tiles;
        kt = at / n;
        return first + at % n;
    }
    // item = position in the list of all parts of a kv head (chunk > 0: there are at most 64 key tiles)
    __device__ void find(int item, int ntk, int& kt, int& part) const {
        const int lane = threadIdx.x & 63;
        int upto = lane < ntk ? parts(lane) : 0;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int below = __shfl_up(upto, o, 64);
            if (lane >= o) upto += below;
        }
        kt = __builtin_amdgcn_readfirstlane(__builtin_popcountll(__builtin_amdgcn_ballot_w64(lane < ntk && upto <= item)));
        part = __builtin_amdgcn_readfirstlane(item - (kt > 0 ? __shfl(upto, kt > 0 ? kt - 1 : 0, 64) : 0));
    }
};
// dS as the dK / dV workgroups leave it for flash_attn_bwd_dq_product_kernel: bf16 blocks of 32 query rows x 32 keys, 2 KB, as
// a wave holds them (store_ds), so that every store of the one and every request of the other is a whole kilobyte.  The
// blocks of 128 query rows are adjacent, ordered by key and then by query row: what a dQ workgroup reads is one stream.
// Only blocks that the causal rule or a window lets be visible have a place.
struct DsBlocks {
    int ntk, causal, window;                         // ntk = tiles of 128 rows (of queries and of keys); window <= rows
    __host__ __device__ int width() const {          // key tiles that have a place for a query tile (causal without a window: qt + 1)
        const int w = causal && window > 0 ? (window - 1 + 127) / 128 + 1 : ntk;
        return w < ntk ? w : ntk;
    }
    __host__ __device__ bool triangle() const { return causal && window <= 0; }
    // first key tile with a place; first block of the query tile
    __host__ __device__ int first(int qt) const { const int f = qt + 1 - width(); return causal && window > 0 && f > 0 ? f : 0; }
    __host__ __device__ int64_t at(int qt) const { return triangle() ? 8 * (int64_t)qt * (qt + 1) : 16 * (int64_t)width() * qt; }
    __host__ __device__ int tiles(int qt) const { return triangle() ? qt + 1 : width(); }
    __host__ __device__ int64_t head_bytes() const { return at(ntk) * 2048; }
};
}  // namespace fab

// CUT: the launch has parts.  (Whole key tiles keep their own instantiation: with the bookkeeping of the parts in the same
// code the pipeline below, which has no register to spare, is 4-8 % slower.)
// OWN_STATS: nothing ran before this kernel, so the workgroup makes the (lse2, delta) pairs of its query rows itself.
// SPILL: dS also goes to `ds`, for the dQ launch after this one.  Under a window that takes 4 and 6 registers more than there are
// (20 and 28 bytes a lane in scratch memory; 2 of CUT without it).
template <int D, bool CAUSAL, AttnMask MASK, bool CUT, bool OWN_STATS, bool SPILL>
__device__ __forceinline__ void bwd_dkv(int block,
    const uint16_t* __restrict__ Q, const uint16_t* __restrict__ Kp, const uint16_t* __restrict__ Vp,
    const uint16_t* __restrict__ O, const uint16_t* __restrict__ dO, const float* __restrict__ LSE, float2* stats,
    uint16_t* __restrict__ dK, uint16_t* __restrict__ dV, int BHkv, int N, int ntk, int npad, float scale, float scale_log2,
    int Hq, int window, const int* __restrict__ kv_lens, const uint8_t* __restrict__ key_mask, fab::Parts plan, int items,
    float* __restrict__ partial, unsigned char* __restrict__ ds) {
    constexpr bool WINDOW = MASK == AttnMask::Limits, PER_KEY = MASK != AttnMask::None;
    if (WINDOW && OWN_STATS && window <= 0) window = INT_MAX;      // lengths alone have no instantiation of their own there
    const int G = plan.G;
    using namespace fab;
    using C = CfgK<D>;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

    const int t = threadIdx.x;
    const int lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int r = lane & 31, g = lane >> 5;

    int bh, item;                         // bh indexes (batch, kv head)
    {
        const bool xcds = (BHkv & 7) == 0;           // heads are dealt to XCDs
        const int heads = xcds ? BHkv >> 3 : BHkv, slot = xcds ? block >> 3 : block;
        if constexpr (CUT) {
            // part after part of all heads, the heaviest first
            bh = slot % heads;
            item = slot / heads;
        } else {
            bh = plan.order(slot, heads, xcds, items, item);
        }
        if (xcds) bh = bh * 8 + (block & 7);
    }
    int kt = item, part = 0;
    if constexpr (CUT) plan.find(item, ntk, kt, part);
    const int n0 = kt * C::BNK;
    const int nw0 = n0 + w * 32;
    const int kvpos = nw0 + r;
    const size_t head_off = (size_t)bh * N * D;                       // of K, V, dK, dV
    const int hkv = Hq / G;
    const size_t qh0 = (size_t)(bh / hkv) * Hq + (size_t)(bh % hkv) * G;   // first query head of the group
    const int Nk = (PER_KEY && kv_lens != nullptr) ? max(0, min(N, kv_lens[bh / hkv])) : N;
    // no key of the block is seen by any query (beyond the length, or all 128 hidden by the key mask)
    bool block_hidden = PER_KEY && n0 >= Nk;
    if (PER_KEY && key_mask != nullptr && !block_hidden) {
        const TileSpan span = visible_tiles(key_mask + (size_t)(bh / hkv) * N + n0, min(C::BNK, Nk - n0), lane);
        block_hidden = span.first >= span.last;
    }
    if constexpr (OWN_STATS) {
        if (!block_hidden) {
            const int first = plan.first(kt), per_head = plan.last(kt) - first, all = G * per_head;
            const int begin = CUT ? part * plan.part_steps(kt) : 0, end = CUT ? min(all, begin + plan.part_steps(kt)) : all;
#pragma unroll 2
            for (int s = 2 * begin + w; s < 2 * end; s += 4) {           // 32 rows a wave, as in the dQ kernel
                const size_t head = qh0 + (s >> 1) / per_head;
                const int qpos = (first + (s >> 1) % per_head) * C::BQ + (s & 1) * 32 + r, qrow = min(qpos, N - 1);
                const size_t off = (head * N + qrow) * D + g * 8;
                float part_sum = 0.0f;
#pragma unroll
                for (int i = 0; i < C::KSTEPS; ++i) part_sum += dot8_bf16(ld_global_16(dO + off + i * 16), ld_global_16(O + off + i * 16));
                const float delta = part_sum + xor32(part_sum);
                float lse2 = LSE[head * N + qrow] * LOG2E;
                if (MASK != AttnMask::None && lse2 == -INFINITY) lse2 = INFINITY;
                if (g == 0) stats[head * npad + qpos] = qpos < N ? make_float2(lse2, delta) : make_float2(INFINITY, 0.0f);
            }
            __threadfence_block();       // before the requests below read the pairs back (other workgroups write equal bytes)
            wait_vmcnt0();
            __syncthreads();
        }
    }

    // ---- this wave's K and V rows as column operands (lane = key row, columns 16i + 8g + [0,8))
    bf16x8 kf[C::KSTEPS], vf[C::KSTEPS];
    {
        const size_t off = head_off + (size_t)min(kvpos, N - 1) * D + g * 8;
#pragma unroll
        for (int i = 0; i < C::KSTEPS; ++i) {
            kf[i] = __builtin_bit_cast(bf16x8, ld_global_16(Kp + off + i * 16));
            vf[i] = __builtin_bit_cast(bf16x8, ld_global_16(Vp + off + i * 16));
        }
    }
    // SPILL: the dS of a hidden key has to be 0, not only what it adds up to here.  Its K and V are taken as 0 and its scores
    // start from -inf instead of 0 (the accumulator operand of their first product), so P and dS are 0 without an instruction
    // in the steps.  Causal launches without a mask have no such key: the ones past N are above every query's diagonal.
    constexpr bool KEY_BIAS = SPILL && (MASK != AttnMask::None || !CAUSAL);
    f32x16 bias;
    if constexpr (KEY_BIAS) {
        const bool hidden = kvpos >= Nk || (key_mask != nullptr && key_mask[(size_t)(bh / hkv) * N + min(kvpos, N - 1)] == 0);
#pragma unroll
        for (int i = 0; i < C::KSTEPS; ++i) {
            const bf16x8 zero = __builtin_bit_cast(bf16x8, u32x4{0, 0, 0, 0});
            kf[i] = hidden ? zero : kf[i];
            vf[i] = hidden ? zero : vf[i];
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) bias[e] = hidden ? -INFINITY : 0.0f;
    }

    // ---- Q / dO / pair tile loaders
    // The G query heads of the group are adjacent in memory: one buffer covers them, a head is a
    // scalar offset.  (Rows past N of a head then alias the next head's first rows instead of
    // reading as zero; their pairs are (+inf, 0), so their probabilities are exactly 0 either way.)
    const uint32_t head_bytes = (uint32_t)N * D * 2u;
    const u32x4 q_rsrc = make_raw_rsrc(Q + qh0 * N * D, head_bytes * (uint32_t)G);
    const u32x4 do_rsrc = make_raw_rsrc(dO + qh0 * N * D, head_bytes * (uint32_t)G);
    const uint32_t stat_bytes = (uint32_t)npad * 8u;
    const u32x4 st_rsrc = make_raw_rsrc(stats + qh0 * npad, stat_bytes * (uint32_t)G);
    constexpr int ROWS_PER_INST = 1024 / C::ROW;
    int g_voff[C::PT];
#pragma unroll
    for (int m = 0; m < C::PT; ++m) {
        const int row = (w * C::PT + m) * ROWS_PER_INST + lane / C::KCH;
        g_voff[m] = row * C::ROW + swz<D>(row, lane % C::KCH) * 16 - 1024 * m;   // request m carries 1024 m as its immediate offset
    }
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
    const uint32_t wave_dst = __builtin_amdgcn_readfirstlane(lds_base + (uint32_t)w * C::PT * 1024u);
    // Tiles past the end of a segment are requested at an offset beyond the buffer (they read as zero), so that
    // every iteration issues the same number of loads and the wait count below stays constant.
    const int jq_first = CAUSAL ? n0 / C::BQ : 0, jq_last = plan.last(kt);      // query tiles that see the block's keys
    // a segment = the tiles [jq0, jq_end) of query head hq of the group
    int hq = 0, jq0 = jq_first, jq_end = jq_last;
    auto issue_tile = [&](int stage, int jq) {
        const uint32_t dst = wave_dst + (uint32_t)stage * C::STAGE;
        const bool live = jq < jq_end;
        const int soff = live ? hq * (int)head_bytes + jq * C::BQ * C::ROW : (int)(head_bytes * (uint32_t)G);
        const int ssoff = live ? (hq * npad + jq * C::BQ) * 8 : (int)(stat_bytes * (uint32_t)G);
        load_global_to_lds_16xN<C::PT>(q_rsrc, dst, g_voff, soff);
        load_global_to_lds_16xN<C::PT>(do_rsrc, dst + C::TILE, g_voff, soff);
        // every wave requests the same kilobyte of pairs (identical bytes, one instruction)
        load_global_to_lds_16(st_rsrc, lds_base + (uint32_t)stage * C::STAGE + 2 * C::TILE, lane * 16, ssoff);
    };

    int row_off[C::KSTEPS];
#pragma unroll
    for (int i = 0; i < C::KSTEPS; ++i) row_off[i] = r * C::ROW + swz<D>(r, 2 * i + g) * 16;
    int tr_lo[C::DT], tr_hi[C::DT];
    {
        const int i16 = lane & 15, b16 = lane >> 4;
        const int row = 4 * (b16 >> 1) + (i16 >> 2);
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt) {
            const int dcol = 32 * dt + 16 * (b16 & 1) + 4 * (i16 & 3);
            tr_lo[dt] = row * C::ROW + swz<D>(row, dcol >> 3) * 16 + (dcol & 7) * 2;
            tr_hi[dt] = (row + 8) * C::ROW + swz<D>(row + 8, dcol >> 3) * 16 + (dcol & 7) * 2;
        }
    }

    f32x16 dk[C::DT], dv[C::DT];
#pragma unroll
    for (int i = 0; i < C::DT; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) { dk[i][e] = 0.0f; dv[i][e] = 0.0f; }

    // LDS addresses.  Inside the pipeline the stage and the sub-tile of every access are
    // compile-time constants, so an address is a per-lane base register plus an immediate; the
    // immediate field holds 16 bits, hence a second set of bases for stages 2 and 3.
    // The bases are made opaque to the compiler, which would otherwise recompute each of them
    // (LDS symbol + offset) next to every use.
    typedef __attribute__((address_space(3))) const unsigned char* lds_cptr;
    auto opaque = [&](int off) {
        uint32_t a = lds_base + (uint32_t)off;
        asm volatile("" : "+v"(a));
        return (lds_cptr)(uintptr_t)a;
    };
    lds_cptr rowp[2][C::KSTEPS], trlo[2][C::DT], trhi[2][C::DT], statp[2];
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
#pragma unroll
        for (int i = 0; i < C::KSTEPS; ++i) rowp[hh][i] = opaque(row_off[i] + hh * 2 * C::STAGE);
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt) {
            trlo[hh][dt] = opaque(tr_lo[dt] + hh * 2 * C::STAGE);
            trhi[hh][dt] = opaque(tr_hi[dt] + hh * 2 * C::STAGE);
        }
        statp[hh] = opaque(2 * C::TILE + 32 * g + hh * 2 * C::STAGE);
    }
    auto tr16 = [](lds_cptr p) {
        typedef __attribute__((ext_vector_type(4))) short s16x4;
        return __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p)));
    };
#define TYR_STG(stg) constexpr int STG = decltype(stg)::value; constexpr int SOFF = (STG & 1) * C::STAGE

    // Row fragments (lane = query row) of sub-tile T of the tile in stage STG
    auto read_rows = [&](auto stg, auto sub, bf16x8 (&qa)[C::KSTEPS], bf16x8 (&da)[C::KSTEPS]) {
        TYR_STG(stg);
        constexpr int T = decltype(sub)::value;
#pragma unroll
        for (int i = 0; i < C::KSTEPS; ++i) {
            lds_cptr p = rowp[STG >> 1][i] + SOFF + T * 32 * C::ROW;
            qa[i] = *reinterpret_cast<__attribute__((address_space(3))) const bf16x8*>(p);
            da[i] = *reinterpret_cast<__attribute__((address_space(3))) const bf16x8*>(p + C::TILE);
        }
    };
    // S = Q K_w^T and dP = dO V_w^T of one sub-tile from its row fragments
    auto scores = [&](const bf16x8 (&qa)[C::KSTEPS], const bf16x8 (&da)[C::KSTEPS], f32x16& s, f32x16& dp) {
#pragma unroll
        for (int e = 0; e < 16; ++e) { s[e] = KEY_BIAS ? bias[e] : 0.0f; dp[e] = 0.0f; }
#pragma unroll
        for (int i = 0; i < C::KSTEPS; ++i) {
            s = mfma_32x32x16_bf16(qa[i], kf[i], s);
            dp = mfma_32x32x16_bf16(da[i], vf[i], dp);
        }
    };
    // P and dS of a sub-tile as column operands.  Register e <-> query row qs0 + 8(e/4) + 4g + e%4;
    // its (lse2, delta) pair sits at pair index 32T + 8(e/4) + 4g + e%4 of the staged kilobyte.
    // Half sh of the pairs of sub-tile T: registers 8sh .. 8sh+7, i.e. k = e/4 in {2sh, 2sh+1}
    auto read_pairs = [&](auto stg, auto sub, auto half, f32x4 (&st)[4]) {
        TYR_STG(stg);
        constexpr int T = decltype(sub)::value, SH = decltype(half)::value;
        lds_cptr St = statp[STG >> 1] + SOFF + 32 * T * 8;
#pragma unroll
        for (int h = 0; h < 2; ++h) {                    // k = 2 SH + h
            st[2 * h] = *reinterpret_cast<__attribute__((address_space(3))) const f32x4*>(St + 8 * (2 * SH + h) * 8);
            st[2 * h + 1] = *reinterpret_cast<__attribute__((address_space(3))) const f32x4*>(St + 8 * (2 * SH + h) * 8 + 16);
        }
    };
    // P and dS of half sh of a sub-tile (query rows qs0 + 16sh + 8h + 4g + x) as one k-step of column operands
    // `apply` (wave-uniform) says whether any (query, key) pair of the rows at hand is hidden from this
    // wave's keys; the mask instructions are skipped otherwise.
    auto probabilities = [&](auto masked, auto half, const f32x4 (&st)[4], int qs0, const f32x16& s, const f32x16& dp,
                             bf16x8& pf, bf16x8& dsf, bool apply) {
        constexpr bool need_mask = decltype(masked)::value;
        constexpr int sh = decltype(half)::value;
        u32x4 ppk, dpk;
#pragma unroll
        for (int h = 0; h < 2; ++h) {                    // e/4 = 2sh + h
            const f32x4 a = st[2 * h];
            const f32x4 b = st[2 * h + 1];
            const float l2[4] = {a[0], a[2], b[0], b[2]};
            const float dl[4] = {a[1], a[3], b[1], b[3]};
            float p[4], ds[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) p[x] = fast_exp2(fmaf(s[8 * sh + 4 * h + x], scale_log2, -l2[x]));
            if (need_mask && apply) {
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    const int qrow = qs0 + 8 * (2 * sh + h) + 4 * g + x;
                    const bool hidden = (CAUSAL && kvpos > qrow) || (WINDOW && qrow - kvpos >= window);
                    if (hidden) p[x] = 0.0f;
                }
            }
#pragma unroll
            for (int x = 0; x < 4; ++x) ds[x] = p[x] * (dp[8 * sh + 4 * h + x] - dl[x]);
            ppk[2 * h] = pack_bf16(p[0], p[1]);
            ppk[2 * h + 1] = pack_bf16(p[2], p[3]);
            dpk[2 * h] = pack_bf16(ds[0], ds[1]);
            dpk[2 * h + 1] = pack_bf16(ds[2], ds[3]);
        }
        pf = __builtin_bit_cast(bf16x8, ppk);
        dsf = __builtin_bit_cast(bf16x8, dpk);
    };
    // Transposed fragments of k-step c = 2T + sh (query rows 16c + 8h + 4g + [0,4)) of dO and Q
    auto read_transposed = [&](auto stg, int c, bf16x8 (&dot)[C::DT], bf16x8 (&qt)[C::DT]) {
        TYR_STG(stg);
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt) {
            lds_cptr pl = trlo[STG >> 1][dt] + SOFF + c * 16 * C::ROW;
            lds_cptr ph = trhi[STG >> 1][dt] + SOFF + c * 16 * C::ROW;
            const bf16x4 lo = tr16(pl + C::TILE);
            const bf16x4 hi = tr16(ph + C::TILE);
            dot[dt] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            const bf16x4 ql = tr16(pl);
            const bf16x4 qh = tr16(ph);
            qt[dt] = __builtin_shufflevector(ql, qh, 0, 1, 2, 3, 4, 5, 6, 7);
        }
    };

    // With WINDOW a step applies the mask only where some pair of the 64 query rows it touches (the second
    // half of u, the first half of u+1) is hidden from this wave's keys: the causal diagonal, the far edge of the window.
    auto rows_are_masked = [&](int qs0) {
        return (CAUSAL && qs0 < nw0 + 32) || (window > 0 && qs0 + 63 - nw0 >= window);
    };
    // dS of half sh of the sub-tile at query row qs0: registers 8 sh .. 8 sh + 7 are query rows 16 sh + 4 g + {0..3} and 8 more.
    // The 16-byte pieces are dealt to the kilobyte so that the transposing reads of the dQ workgroup, which take the same key
    // of both halves and both g at once, find them in different banks.
    const fab::DsBlocks place{ntk, CAUSAL, WINDOW ? window : 0};
    unsigned char* ds_head = nullptr;
    const uint32_t ds_lane[2] = {(uint32_t)(g * 32 + (r ^ (4 * g))) * 16u, (uint32_t)(g * 32 + (r ^ (4 * g + 8))) * 16u + 1024u};
    auto store_ds = [&](int sh, int qs0, bf16x8 v) {
        const int qt = qs0 >> 7;
        unsigned char* to = ds_head + (place.at(qt) + (4 * (kt - place.first(qt)) + w) * 4 + ((qs0 >> 5) & 3)) * 2048;
        st_global_16(to + ds_lane[sh], __builtin_bit_cast(u32x4, v));
    };
    bf16x8 rq[C::KSTEPS], rd[C::KSTEPS];              // row fragments of the next sub-tile, read one step ahead
    bf16x8 pf0, dsf0;                                 // P, dS of the first half of the current sub-tile
    f32x4 st1[4];                                     // pairs of its second half
    using Half0 = std::integral_constant<int, 0>;
    using Half1 = std::integral_constant<int, 1>;
    // One step of the software pipeline on sub-tile u = 2t + T, tile t in stage STG (scores in sc / dpc).
    // With one wave per SIMD a vector instruction overlaps with the matrix pipe only where it sits
    // between two MFMAs of the wave's own stream, and the pipe idles through any stretch of vector
    // work that is longer than the MFMA before it.  The step therefore has two phases of 16 MFMAs,
    // each carrying half a sub-tile's exponentials:
    //   A: S, dP of sub-tile u+1 (row fragments already in rq / rd)  beside  P, dS of the second half of u
    //   B: dV, dK of u (both halves)                                  beside  P, dS of the first half of u+1
    // so that P, dS of a sub-tile's first half are always computed one step ahead (pf0 / dsf0).
    // The row fragments of u+2 and the pairs of u+1 are requested a phase before they are used.
    // Past the last sub-tile the "next" reads hit a stage without live data; their results are dropped.
    auto step = [&](auto masked, auto stg, auto sub, int qs0, f32x16& sc, f32x16& dpc, f32x16& sn, f32x16& dpn) {
        constexpr int STG = decltype(stg)::value, T = decltype(sub)::value;
        using Stg1 = std::integral_constant<int, T == 0 ? STG : ((STG + 1) & 3)>;       // stage of u+1
        using Sub1 = std::integral_constant<int, 1 - T>;
        using Stg2 = std::integral_constant<int, (STG + 1) & 3>;                        // stage of u+2
        bf16x8 dot0[C::DT], qt0[C::DT], dot1[C::DT], qt1[C::DT];
        f32x4 st0[4];
        if constexpr (SPILL) store_ds(0, qs0, dsf0);
        read_transposed(stg, 2 * T, dot0, qt0);
        read_pairs(Stg1{}, Sub1{}, Half0{}, st0);
        read_transposed(stg, 2 * T + 1, dot1, qt1);
        scores(rq, rd, sn, dpn);
        bf16x8 pf1, dsf1;
        const bool apply = decltype(masked)::value && rows_are_masked(qs0);       // rows qs0 .. qs0 + 63
        probabilities(masked, Half1{}, st1, qs0, sc, dpc, pf1, dsf1, apply);
        if constexpr (SPILL) store_ds(1, qs0, dsf1);
        read_pairs(Stg1{}, Sub1{}, Half1{}, st1);          // ahead of the row fragments: LDS answers in order
        read_rows(Stg2{}, sub, rq, rd);
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt) {
            dv[dt] = mfma_32x32x16_bf16(dot0[dt], pf0, dv[dt]);
            dk[dt] = mfma_32x32x16_bf16(qt0[dt], dsf0, dk[dt]);
        }
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt) {
            dv[dt] = mfma_32x32x16_bf16(dot1[dt], pf1, dv[dt]);
            dk[dt] = mfma_32x32x16_bf16(qt1[dt], dsf1, dk[dt]);
        }
        probabilities(masked, Half0{}, st0, qs0 + 32, sn, dpn, pf0, dsf0, apply);
#ifndef TYR_DKV_NO_SCHED
        // issue order: one MFMA, then its share of the LDS reads and of the vector work
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
            __builtin_amdgcn_sched_group_barrier(0x400, 1, 0);
        }
#pragma unroll
        for (int i = 0; i < 12; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
            __builtin_amdgcn_sched_group_barrier(0x400, 1, 0);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
            __builtin_amdgcn_sched_group_barrier(0x400, 1, 0);
        }
#endif
    };
    // What a step expects of the step before it, for the wave's first sub-tile: its scores, P and dS
    // of its first half, the pairs of its second half, and the row fragments of the sub-tile after
    // it.  Without WINDOW the only partially masked sub-tile of a causal wave is this one (its
    // diagonal): hidden scores become -inf here, which the steps turn into P = 0 and dS = 0 like any
    // other score, so they carry no mask instructions.
    auto first_scores = [&](auto masked, auto stg, auto sub, int qs0, f32x16& sc, f32x16& dpc) {
        constexpr int STG = decltype(stg)::value, T = decltype(sub)::value;
        using Stg1 = std::integral_constant<int, T == 0 ? STG : ((STG + 1) & 3)>;     // stage of u+1
        using Sub1 = std::integral_constant<int, 1 - T>;
        f32x4 st0[4];
        read_rows(stg, sub, rq, rd);
        read_pairs(stg, sub, Half0{}, st0);
        read_pairs(stg, sub, Half1{}, st1);
        scores(rq, rd, sc, dpc);
        if (CAUSAL && !WINDOW) {
#pragma unroll
            for (int e = 0; e < 16; ++e)
                if (kvpos > qs0 + 8 * (e >> 2) + 4 * g + (e & 3)) sc[e] = -INFINITY;
        }
        read_rows(Stg1{}, Sub1{}, rq, rd);
        probabilities(masked, Half0{}, st0, qs0, sc, dpc, pf0, dsf0, true);
    };
#undef TYR_STG

#pragma unroll
    for (int i = 0; i < C::KSTEPS; ++i) { pin_registers(kf[i]); pin_registers(vf[i]); }
    // this part's steps of the block; a block that no query sees has none (its rows are 0)
    const int per_head = jq_last - jq_first, per_part = CUT ? plan.part_steps(kt) : 0;
    if constexpr (SPILL && MASK == AttnMask::Keys) {
        // all 128 keys hidden between visible ones: the dQ workgroups walk from the first visible key to the last
        if (block_hidden && key_mask != nullptr) {
            const TileSpan span = visible_tiles(key_mask + (size_t)(bh / hkv) * N, N, lane);
            const int all = G * per_head, end = CUT ? min(all, (part + 1) * per_part) : all;
            if (span.first < 2 * kt + 2 && span.last > 2 * kt)
                for (int at = CUT ? part * per_part : 0; at < end; ++at) {
                    ds_head = ds + (size_t)(qh0 + at / per_head) * place.head_bytes();
                    for (int qs0 = (jq_first + at % per_head) * C::BQ, T = 0; T < 2; ++T, qs0 += 32)
                        if (!CAUSAL || qs0 >= nw0)
                            for (int sh = 0; sh < 2; ++sh) store_ds(sh, qs0, __builtin_bit_cast(bf16x8, u32x4{0, 0, 0, 0}));
                }
        }
    }
    const int step_end = block_hidden ? 0 : CUT ? min(G * per_head, (part + 1) * per_part) : G;
    for (int step_at = CUT ? part * per_part : 0; step_at < step_end;) {
    if constexpr (CUT) {
        hq = step_at / per_head;
        jq0 = jq_first + step_at % per_head;
        jq_end = min(jq_last, jq0 + step_end - step_at);
        step_at += jq_end - jq0;
    } else {
        hq = step_at++;
    }
    if constexpr (SPILL) ds_head = ds + (size_t)(qh0 + hq) * place.head_bytes();
    const int ntile = jq_end - jq0;
    const int nsub = 2 * ntile;                       // 32-row sub-tiles, numbered from the segment's first tile
    // First sub-tile with a visible (query, key) pair for this wave.  Causal: the block's first
    // tile starts at query n0 and the wave's keys at n0 + 32w, so sub-tile w of the head is the wave's diagonal
    // one (the only partially masked one); earlier sub-tiles are skipped.
    const int u0 = !CAUSAL ? 0 : CUT ? max(0, w - 2 * (jq0 - jq_first)) : w;
    issue_tile(0, jq0);
    issue_tile(1, jq0 + 1);
    issue_tile(2, jq0 + 2);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * C::LOADS_PER_TILE) : "memory");
    __syncthreads();

    // Tile t+1 is awaited, and tile t+3 requested into the stage tile t-1 has left, before the
    // first sub-tile of tile t (whose steps already read fragments of tile t+1): four stages.
    // SPILL: a step's two stores count as well; tile t+1 was requested before the stores of the last two tiles, if these
    // were steps of this wave (it skips the first u0), and before tile t+2.
    auto tile_boundary = [&](int u) {
        if (!(u & 1) && (u >> 1) + 1 < ntile) {
            if (SPILL && u - u0 >= 4) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::LOADS_PER_TILE + 8) : "memory");
            else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::LOADS_PER_TILE) : "memory");
            __syncthreads();
            issue_tile(((u >> 1) + 3) & (C::NST - 1), jq0 + (u >> 1) + 3);
        }
    };
    using std::integral_constant;
    using MaskedT = integral_constant<bool, WINDOW>;
    const int qbase = jq0 * C::BQ;
    // Scores ping-pong between two register sets by the parity of u (no copies).
    f32x16 sA, dpA, sB, dpB;
    int u = 0;
    for (; u < u0 && u < nsub; ++u) tile_boundary(u);           // sub-tiles above the wave's diagonal
    if (u < nsub) {
        // u = u0 < 4: stage u0 / 2, sub-tile u0 % 2; even sub-tiles keep their scores in sA / dpA
        switch (u) {
            case 0:  first_scores(MaskedT{}, integral_constant<int, 0>{}, integral_constant<int, 0>{}, qbase, sA, dpA); break;
            case 1:  first_scores(MaskedT{}, integral_constant<int, 0>{}, integral_constant<int, 1>{}, qbase + 32, sB, dpB); break;
            case 2:  first_scores(MaskedT{}, integral_constant<int, 1>{}, integral_constant<int, 0>{}, qbase + 64, sA, dpA); break;
            default: first_scores(MaskedT{}, integral_constant<int, 1>{}, integral_constant<int, 1>{}, qbase + 96, sB, dpB); break;
        }
    }
    // the pipeline, unrolled over the 8 (stage, sub-tile) combinations; entered at u % 8
#define TYR_STEP(K, CS, CD, NS, ND)                                                                          \
    case K:                                                                                                  \
        if (u >= nsub) goto pipeline_done;                                                                   \
        tile_boundary(u);                                                                                    \
        step(MaskedT{}, integral_constant<int, (K) / 2>{},                                                   \
             integral_constant<int, (K) % 2>{}, qbase + 32 * u, CS, CD, NS, ND);                             \
        ++u;                                                                                                 \
        [[fallthrough]];
    for (;;) {
        switch (u & 7) {
            TYR_STEP(0, sA, dpA, sB, dpB)
            TYR_STEP(1, sB, dpB, sA, dpA)
            TYR_STEP(2, sA, dpA, sB, dpB)
            TYR_STEP(3, sB, dpB, sA, dpA)
            TYR_STEP(4, sA, dpA, sB, dpB)
            TYR_STEP(5, sB, dpB, sA, dpA)
            TYR_STEP(6, sA, dpA, sB, dpB)
            TYR_STEP(7, sB, dpB, sA, dpA)
            default: break;
        }
    }
pipeline_done:
#undef TYR_STEP
    wait_vmcnt0();                                   // drain before the next segment reuses the stages
    __syncthreads();
    }

    if constexpr (PER_KEY) {
        if (kvpos >= Nk || (key_mask != nullptr && key_mask[(size_t)(bh / hkv) * N + min(kvpos, N - 1)] == 0)) {
#pragma unroll
            for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
                for (int e = 0; e < 16; ++e) dv[dt][e] = dk[dt][e] = 0.0f;
        }
    }
    if (CUT && plan.parts(kt) > 1) {
        // [2 (dV, dK)][wave][register group of four][lane] f32x4: coalesced as the accumulators lie
        f32x4* out = reinterpret_cast<f32x4*>(partial) + ((size_t)bh * items + item) * (2 * 4 * C::DT * 4 * 64) + w * (C::DT * 4 * 64) + lane;
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                out[(dt * 4 + q4) * 64] = f32x4{dv[dt][4 * q4], dv[dt][4 * q4 + 1], dv[dt][4 * q4 + 2], dv[dt][4 * q4 + 3]};
                out[(4 * C::DT * 4 + dt * 4 + q4) * 64] = f32x4{dk[dt][4 * q4], dk[dt][4 * q4 + 1], dk[dt][4 * q4 + 2], dk[dt][4 * q4 + 3]};
            }
        return;
    }
    unsigned char* scratch = lds + w * (32 * (D * 2 + 16));
    store_transposed_bf16<D>(dv, 1.0f, scratch, dV + head_off + (size_t)nw0 * D, N - nw0, lane);
    store_transposed_bf16<D>(dk, scale, scratch, dK + head_off + (size_t)nw0 * D, N - nw0, lane);
}

template <int D, bool CAUSAL, AttnMask MASK, bool CUT, bool SPILL>
__global__ __launch_bounds__(fab::THREADS, 1) void flash_attn_bwd_dkv_kernel(
    const uint16_t* __restrict__ Q, const uint16_t* __restrict__ Kp, const uint16_t* __restrict__ Vp,
    const uint16_t* __restrict__ dO, float2* stats, uint16_t* __restrict__ dK, uint16_t* __restrict__ dV, int BHkv, int N,
    int ntk, int npad, float scale, float scale_log2, int Hq, int window, const int* __restrict__ kv_lens,
    const uint8_t* __restrict__ key_mask, fab::Parts plan, int items, float* __restrict__ partial, unsigned char* __restrict__ ds) {
    bwd_dkv<D, CAUSAL, MASK, CUT, false, SPILL>(blockIdx.x, Q, Kp, Vp, nullptr, dO, nullptr, stats, dK, dV, BHkv, N, ntk, npad, scale, scale_log2,
                                         Hq, window, kv_lens, key_mask, plan, items, partial, ds);
}

// ------------------------------------------------------------------------------------------
// dK, dV of 256 keys for launches of many whole key tiles (after a dQ launch that has left the statistics of the rows in groups
// of four): 4 waves of 64 keys, each over all rows of every query tile.
//
// One wave a SIMD, so what a wave issues between two products is what bounds it, and LDS reads are the dearest of that (an
// instruction every 5 ns and wave).  With 64 keys a wave instead of bwd_dkv's 32, each fragment read serves twice the products,
// and what a workgroup takes to start and end (14 us) is paid half as often.  That takes all 512 registers: the 256
// accumulation registers are dK and dV of 64 x 128, K and V fragments 128 of the others.  Scores come in sub-tiles of 16 query
// rows by 16x16x32 products, whose results take half the registers of 32x32 ones; a row exchange (v_permlane16_swap)
// makes P and dS of two of their 16-key blocks the column operand of a 32x32x16 product.  All products are in asm: the compiler has all results
// of its own in accumulation registers here, or none, and copies the others back and forth.
// dK/dV by bwd_dkv and by this: B16 H16 N4096 causal 2232 and 1850 us, at D = 64 1370 and 1170; B8 H16 N4096 not causal 2050 and 1600.
namespace fab {
// The bank swizzle for row fragments of 16 rows x 64 bytes.  A 16-byte LDS read serves lanes {0-3, 12-15, 20-27} at once, then
// {4-11, 16-19, 28-31}: rows 0-3 and 12-15 of one chunk with rows 4-11 of the next (rows of the product; as query rows, bits 2 and 3
// are exchanged).  The two low bits keep those apart (SQ_LDS_BANK_CONFLICT 0.3 of the LDS cycles with swz, none so); the upper ones are swz's.
template <int D> __device__ __forceinline__ int swz16(int row, int c) {
    const int low = (((row >> 3) ^ (row >> 2)) & 1) << 1 | ((row >> 2) & 1);
    return c ^ ((D == 128 ? (row & 3) << 2 : ((row >> 1) & 1) << 2) | low);
}
// Scalar offset of the request for piece m (4 KB) of the query tile at `tile` in a buffer of `bytes`: never beyond the buffer, like every
// request's here.  (The range check is on the whole offset; the manual gives it as lane offset >= bytes - scalar offset, and does not
// say what a scalar offset above bytes makes of the difference.)  A piece that would start there has no row of the buffer.
__host__ __device__ inline uint32_t piece_at(uint32_t tile, int m, uint32_t bytes) {
    const uint32_t at = tile + 4096u * m;            // (both below 2^31)
    return at < bytes ? at : bytes;
}
// P and dS of a lane (slot j <-> query row 8 (j / 4) + j % 4) set to 0 where gap + that row is not below `seen`
__device__ __forceinline__ void clear_hidden_pairs(uint32_t gap, uint32_t seen, bf16x8& p, bf16x8& d) {
    u32x4 keep;
#pragma unroll
    for (int y = 0; y < 4; ++y) {
        const uint32_t row = 8 * (y >> 1) + 2 * (y & 1);
        keep[y] = (gap + row < seen ? 0xffffu : 0u) | (gap + row + 1 < seen ? 0xffff0000u : 0u);
    }
    p = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, p) & keep);
    d = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, d) & keep);
}
}  // namespace fab

template <int D, bool CAUSAL, AttnMask MASK>
__global__ __launch_bounds__(fab::THREADS, 1) void flash_attn_bwd_dkv_wide_kernel(
    const uint16_t* __restrict__ Q, const uint16_t* __restrict__ Kp, const uint16_t* __restrict__ Vp,
    const uint16_t* __restrict__ dO, const float2* __restrict__ stats, uint16_t* __restrict__ dK, uint16_t* __restrict__ dV, int BHkv, int N,
    int npad, float scale, float scale_log2, int Hq, int window, const int* __restrict__ kv_lens,
    const uint8_t* __restrict__ key_mask, fab::Parts plan, int items) {
    constexpr bool WINDOW = MASK == AttnMask::Limits, PER_KEY = MASK != AttnMask::None;
    constexpr int BNK = 256, NSUB = 4;               // keys of the workgroup; 16-row sub-tiles of a query tile
    const int G = plan.G;
    using namespace fab;
    using C = CfgK<D>;
    constexpr int KS = D / 32;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

    const int t = threadIdx.x;
    const int lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l16 = lane & 15, g4 = lane >> 4;

    const bool xcds = (BHkv & 7) == 0;               // heads are dealt to XCDs
    int kt;
    int bh = plan.order(xcds ? blockIdx.x >> 3 : blockIdx.x, xcds ? BHkv >> 3 : BHkv, xcds, items, kt);
    bh = __builtin_amdgcn_readfirstlane(xcds ? bh * 8 + (int)(blockIdx.x & 7) : bh);        // of (batch, kv head)
    kt = __builtin_amdgcn_readfirstlane(kt);
    const int n0 = kt * BNK;
    const int nw0 = n0 + 64 * w;                                      // this wave's first key
    const size_t head_off = (size_t)bh * N * D;                       // of K, V, dK, dV
    const int hkv = Hq / G;
    const size_t qh0 = (size_t)(bh / hkv) * Hq + (size_t)(bh % hkv) * G;   // first query head of the group
    const int Nk = (PER_KEY && kv_lens != nullptr) ? max(0, min(N, kv_lens[bh / hkv])) : N;
    // no key of the block is seen by any query (beyond the length, or all hidden by the key mask)
    bool block_hidden = PER_KEY && n0 >= Nk;
    if (PER_KEY && key_mask != nullptr && !block_hidden) {
        const TileSpan span = visible_tiles(key_mask + (size_t)(bh / hkv) * N + n0, min(BNK, Nk - n0), lane);
        block_hidden = span.first >= span.last;
    }
    // the query tiles that see the block's keys, head after head of the group
    const int jq_first = plan.first(kt), jq_last = __builtin_amdgcn_readfirstlane(plan.last(kt));
    const int ntile = __builtin_amdgcn_readfirstlane(block_hidden ? 0 : G * (jq_last - jq_first));

    // ---- Q / dO / statistics loaders
    // The G query heads of the group are adjacent in memory: one buffer covers them, a head is a
    // scalar offset.  (Rows past N of a head then alias the next head's first rows instead of
    // reading as zero; their statistics are (+inf, 0), so their probabilities are exactly 0 either way.)
    const uint32_t head_bytes = (uint32_t)N * D * 2u, group_bytes = head_bytes * (uint32_t)G;
    const u32x4 q_rsrc = make_raw_rsrc(Q + qh0 * N * D, group_bytes);
    const u32x4 do_rsrc = make_raw_rsrc(dO + qh0 * N * D, group_bytes);
    const uint32_t stat_bytes = (uint32_t)npad * 8u;
    const u32x4 st_rsrc = make_raw_rsrc(stats + qh0 * npad, stat_bytes * (uint32_t)G);
    // Request m of a wave fills the kilobyte at 4 KB m + 1 KB w of a tile: the rows of one swizzle, so that one register of
    // per-lane offsets serves all of them.
    static_assert(C::PT * 4096 == C::TILE, "a request of each of four waves is 4 KB");
    int g_voff;
    {
        const int row = w * (1024 / C::ROW) + lane / C::KCH;
        g_voff = row * C::ROW + swz16<D>(row, lane % C::KCH) * 16;
    }
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
    const uint32_t wave_dst = __builtin_amdgcn_readfirstlane(lds_base + (uint32_t)w * 1024u);
    // Query tile `rq_jq` of head `rq_head`, piece by piece.  Tiles past the last are requested at the buffer's
    // end (they read as zero), so that every iteration issues the same number of loads and the wait count below stays constant.
    int rq_head = 0, rq_jq = jq_first, rq_left = ntile;
    int rq_at = 0, rq_stats_at = 0;                  // offsets of the tile that is being requested
    auto request_begin = [&] {
        rq_at = __builtin_amdgcn_readfirstlane(rq_left > 0 ? rq_head * (int)head_bytes + rq_jq * C::BQ * C::ROW : (int)group_bytes);
        rq_stats_at = __builtin_amdgcn_readfirstlane(rq_left > 0 ? (rq_head * npad + rq_jq * C::BQ) * 8 : (int)(stat_bytes * (uint32_t)G));
        --rq_left;
        if (++rq_jq == jq_last) { rq_jq = jq_first; ++rq_head; }
    };
    auto request_piece = [&](int stage, int m) {
        const uint32_t dst = wave_dst + (uint32_t)stage * C::STAGE + 4096u * m;
        const int at = (int)piece_at((uint32_t)rq_at, m, group_bytes);
        load_global_to_lds_16(q_rsrc, dst, g_voff, at);
        load_global_to_lds_16(do_rsrc, dst + C::TILE, g_voff, at);
    };
    // every wave requests the same kilobyte of statistics (identical bytes, one instruction)
    auto request_stats = [&](int stage) {
        load_global_to_lds_16(st_rsrc, lds_base + (uint32_t)stage * C::STAGE + 2 * C::TILE, lane * 16, rq_stats_at);
    };
    auto request_tile = [&](int stage) {
        request_begin();
#pragma unroll
        for (int m = 0; m < C::PT; ++m) request_piece(stage, m);
        request_stats(stage);
    };

    // The first query tile is on its way before K and V are, the others behind them; everything is waited for at once.
    if (ntile > 0) request_tile(0);
    // ---- this wave's K and V rows as column operands (lane = key row 16b + l%16, columns 32i + 8(l/16) + [0,8))
    bf16x8 kf[4][KS], vf[4][KS];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const size_t off = head_off + (size_t)min(nw0 + 16 * b + l16, N - 1) * D + g4 * 8;
#pragma unroll
        for (int i = 0; i < KS; ++i) {
            kf[b][i] = __builtin_bit_cast(bf16x8, ld_global_16(Kp + off + i * 32));
            vf[b][i] = __builtin_bit_cast(bf16x8, ld_global_16(Vp + off + i * 32));
        }
    }
    if (ntile > 0) {
        request_tile(1);
        request_tile(2);
    }

    // LDS addresses, of stage 0; the loop moves them from stage to stage.  Row i of a score product is query row pi(i) of
    // the sub-tile, bits 2 and 3 of i exchanged: the row exchange then leaves P and dS with lane half g holding query rows
    // 4g + {0..3} and 4g + 8 + {0..3}, which is what the transposing reads of Q and dO deliver.
    // (A chunk of 64 columns further is a flip of bit 6 and up: swz16 and the rows' alignment.)
    const int row16 = (l16 & 3) | ((l16 & 4) << 1) | ((l16 & 8) >> 1);
    const int q4 = ((g4 & 1) << 3) | ((g4 & 2) << 1);              // first of the four query rows of a lane's scores
    uint32_t rowp, trlo, trhi, statp;
    {
        const int trow = 4 * (g4 >> 1) + (l16 >> 2), tcol = 16 * (g4 & 1) + 4 * (l16 & 3);
        rowp = lds_base + row16 * C::ROW + swz16<D>(row16, g4) * 16;
        trlo = lds_base + trow * C::ROW + swz16<D>(trow, tcol >> 3) * 16 + (tcol & 7) * 2;
        trhi = lds_base + (trow + 8) * C::ROW + swz16<D>(trow + 8, tcol >> 3) * 16 + (tcol & 7) * 2;
        statp = lds_base + 2 * C::TILE + q4 * 8;
    }
    typedef __attribute__((address_space(3))) const unsigned char* lds_cptr;
    auto read_row = [](uint32_t a) { return *reinterpret_cast<__attribute__((address_space(3))) const bf16x8*>((lds_cptr)(uintptr_t)a); };
    auto read_stats = [](uint32_t a) { return *reinterpret_cast<__attribute__((address_space(3))) const f32x4*>((lds_cptr)(uintptr_t)a); };
    auto tr16 = [](uint32_t a) {
        typedef __attribute__((ext_vector_type(4))) short s16x4;
        return __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(uintptr_t)a));
    };

    f32x16 dk[C::DT][2], dv[C::DT][2];               // [32 columns of D][32 keys]
#pragma unroll
    for (int i = 0; i < C::DT; ++i)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int e = 0; e < 16; ++e) { dk[i][b][e] = 0.0f; dv[i][b][e] = 0.0f; }

    f32x4 s[4], dp[4];                               // scores and dP - delta of 16 query rows x 16 keys, register x <-> query row q4 + x
    bf16x8 pf[2], dsf[2];                            // P and dS of the sub-tile at hand as column operands of 32 keys
    bf16x8 fq[KS], fd[KS];                           // row fragments of Q and dO, of the next sub-tile
    f32x4 neg_delta;                                 // of the lane's rows of the next sub-tile: what dP starts from
    auto read_rows = [&](int i, int off) {
        fq[i] = read_row((rowp ^ (64 * i)) + off);
        fd[i] = read_row((rowp ^ (64 * i)) + off + C::TILE);
    };
    // S = Q K^T and dP - delta = dO V^T - delta of a sub-tile: k-step i, keys 16b + {0..15}
    auto scores = [&](int i, int b) {
        if (i == 0) {
            mfma_16x16x32_bf16_vgpr_begin(s[b], fq[i], kf[b][i]);
            mfma_16x16x32_bf16_vgpr_begin(dp[b], fd[i], vf[b][i], neg_delta);
        } else {
            mfma_16x16x32_bf16_vgpr(s[b], fq[i], kf[b][i]);
            mfma_16x16x32_bf16_vgpr(dp[b], fd[i], vf[b][i]);
        }
    };
    // P and dS of the scores in 16 pieces of vector instructions, with slot(0) .. slot(15) behind them
    auto probabilities = [&](const f32x4& lse2, bf16x8 (&p_out)[2], bf16x8 (&ds_out)[2], auto&& slot) {
        u32x2 pp[2], dd[2];
        u32x4 po, dso;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            float p[4], d[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) p[x] = fmaf(s[b][x], scale_log2, -lse2[x]);
            slot(4 * b);
#pragma unroll
            for (int x = 0; x < 4; ++x) p[x] = fast_exp2(p[x]);
            slot(4 * b + 1);
#pragma unroll
            for (int x = 0; x < 4; ++x) d[x] = p[x] * dp[b][x];
            slot(4 * b + 2);
            pp[b & 1] = u32x2{pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3])};
            dd[b & 1] = u32x2{pack_bf16(d[0], d[1]), pack_bf16(d[2], d[3])};
            if (b & 1) {
                // lane groups (0, 1, 2, 3) of two 16-key blocks -> (0, 0', 2, 2') and (1, 1', 3, 3')
#pragma unroll
                for (int y = 0; y < 2; ++y) {
                    const u32x2 sp = __builtin_amdgcn_permlane16_swap(pp[0][y], pp[1][y], false, false);
                    const u32x2 sd = __builtin_amdgcn_permlane16_swap(dd[0][y], dd[1][y], false, false);
                    po[y] = sp.x; po[2 + y] = sp.y;
                    dso[y] = sd.x; dso[2 + y] = sd.y;
                }
                p_out[b >> 1] = __builtin_bit_cast(bf16x8, po);
                ds_out[b >> 1] = __builtin_bit_cast(bf16x8, dso);
            }
            slot(4 * b + 3);
        }
    };
    // Hidden pairs of the sub-tile at query row q0, if it has any (wave-uniform): P = dS = 0, whatever was computed for them.
    // A pair is visible iff 0 <= query - key < window; `gap` is query - key of the lane's first query row at q0 = 0.
    const uint32_t gap = (uint32_t)(4 * (lane >> 5) - nw0 - (lane & 31));
    const uint32_t seen = WINDOW ? (uint32_t)window : 0x80000000u;
    auto hide = [&](int q0, bf16x8 (&p)[2], bf16x8 (&d)[2]) {
        if constexpr (CAUSAL) {
            if (__builtin_expect(q0 < nw0 + 63 || (WINDOW && q0 + 15 - nw0 >= window), 0)) {
                clear_hidden_pairs(gap + (uint32_t)q0, seen, p[0], d[0]);
                clear_hidden_pairs(gap + (uint32_t)q0 - 32u, seen, p[1], d[1]);
            }
        }
    };

    if (ntile > 0) {
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < KS; ++i) { pin_registers(kf[b][i]); pin_registers(vf[b][i]); }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * C::LOADS_PER_TILE) : "memory");
    __syncthreads();

    // Sub-tile 0 up to P and dS, and the row fragments of sub-tile 1: what a step finds of its predecessor.
    neg_delta = read_stats(statp + 16);
#pragma unroll
    for (int i = 0; i < KS; ++i) {
        read_rows(i, 0);
#pragma unroll
        for (int b = 0; b < 4; ++b) scores(i, b);
        if (i == 1) asm volatile("" ::"v"(neg_delta));
        __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_nop 7" : "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]), "+v"(dp[0]), "+v"(dp[1]), "+v"(dp[2]), "+v"(dp[3]));
    probabilities(read_stats(statp), pf, dsf, [](int) { __builtin_amdgcn_sched_barrier(0); });
    int jq = jq_first;                               // the tile at hand
    hide(jq * C::BQ, pf, dsf);
#pragma unroll
    for (int i = 0; i < KS - 1; ++i) read_rows(i, 16 * C::ROW);
    neg_delta = read_stats(statp + 128 + 16);

    // A step on sub-tile u of a tile has two phases of as many matrix cycles:
    //   A: S and dP of u + 1, beside the transposed fragments of u and a piece of the request for the tile after next but one
    //   B: dV and dK of u, beside P and dS of u + 1 and the row fragments of u + 2
    // The vector work of B fits between its 32x32x16 products; the fences keep the order that is written here (the compiler
    // does not know that the asm is products).  `advance` moves an address to the next stage of the ring; q0 is the first row of u + 1.
    auto step = [&](auto sub, int advance, int into, int q0) {
        constexpr int SUB = decltype(sub)::value, NEXT = (SUB + 1) % NSUB, NEXT2 = (SUB + 2) % NSUB;
        constexpr int OFF = SUB * 16 * C::ROW;
        bf16x4 tr[C::DT][4];                         // of dO: query rows 4g + {0..3} and 8 more; of Q
        auto read_transposed = [&](int piece) {
            const int dt = piece >> 2, x = piece & 3;
            tr[dt][x] = tr16((((x & 1) ? trhi : trlo) ^ (64 * dt)) + OFF + (x < 2 ? C::TILE : 0));
        };
        f32x4 lse2;
        if (SUB == 0) request_begin();
#pragma unroll
        for (int i = 0; i < KS; ++i)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int at = 4 * i + b;            // two products, then their share of the rest
                scores(i, b);
                if (at < 4 * (C::DT - 1)) read_transposed(at);
                if (at == 1) read_rows(KS - 1, NEXT * 16 * C::ROW);
                if (at == 4 * KS - 5) lse2 = read_stats(statp + NEXT * 128);
                if (at == 2 && SUB < C::PT) request_piece(into, SUB);
                if (SUB == 0 && at == 4 * KS - 1) request_stats(into);
                if (at == 7) asm volatile("" ::"v"(neg_delta));      // no other use of its registers while products read them
                __builtin_amdgcn_sched_barrier(0);
            }
        if (SUB == NSUB - 2) { rowp += advance; statp += advance; }
        bf16x8 pn[2], dsn[2];
        // product m: dV and dK in turn, columns m / 4 of D, keys (m / 2) % 2
        auto product = [&](int m) {
            const int dt = m >> 2, b = (m >> 1) & 1, x = 2 * (m & 1);
            const bf16x8 f = __builtin_shufflevector(tr[dt][x], tr[dt][x + 1], 0, 1, 2, 3, 4, 5, 6, 7);
            if (m & 1) mfma_32x32x16_bf16_acc(dk[dt][b], f, dsf[b]); else mfma_32x32x16_bf16_acc(dv[dt][b], f, pf[b]);
        };
        // Wait states between an ordinary instruction and a product on its result (P, dS), and between a product and an ordinary
        // instruction on its result: the first scores are used behind product(0), eight products and this after their own.
        asm volatile("s_nop 1" : "+v"(pf[0]), "+v"(pf[1]), "+v"(dsf[0]), "+v"(dsf[1]), "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]),
                     "+v"(dp[0]), "+v"(dp[1]), "+v"(dp[2]), "+v"(dp[3]));
        product(0);
        __builtin_amdgcn_sched_barrier(0);
        probabilities(lse2, pn, dsn, [&](int k) {
            if (k < 4) read_transposed(4 * (C::DT - 1) + k);
            if (k + 1 < 4 * C::DT) product(k + 1);
            if (k >= 8 && !(k & 1) && (k - 8) / 2 < KS - 1) read_rows((k - 8) / 2, NEXT2 * 16 * C::ROW);
            if (k == 13) neg_delta = read_stats(statp + NEXT2 * 128 + 16);
            __builtin_amdgcn_sched_barrier(0);
        });
        hide(q0, pn, dsn);
        if (SUB == NSUB - 1) { trlo += advance; trhi += advance; }
#pragma unroll
        for (int b = 0; b < 2; ++b) { pf[b] = pn[b]; dsf[b] = dsn[b]; }
    };
    // Tile t+1 is awaited, and tile t+3 requested into the stage tile t-1 has left, before and in the steps of tile t (which read
    // row fragments of tile t+1): four stages.  (No wait for LDS reads in front of the barrier, as __syncthreads would have: the ones
    // on their way are of tile t, those of tile t-1 have all been used.)
    int stage = 0;
    for (int tile = 0; tile < ntile; ++tile) {
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(C::LOADS_PER_TILE) : "memory");
        const int into = (stage + 3) & (C::NST - 1);
        const int advance = stage == C::NST - 1 ? -(C::NST - 1) * C::STAGE : C::STAGE;
        const int q0 = jq * C::BQ;
        step(std::integral_constant<int, 0>{}, advance, into, q0 + 16);
        step(std::integral_constant<int, 1>{}, advance, into, q0 + 32);
        step(std::integral_constant<int, 2>{}, advance, into, q0 + 48);
        if (++jq == jq_last) jq = jq_first;
        step(std::integral_constant<int, 3>{}, advance, into, jq * C::BQ);
        stage = (stage + 1) & (C::NST - 1);
    }
    }
    // (the wait states between a product and an ordinary instruction on its result)
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt)
        asm volatile("" : "+a"(dk[dt][0]), "+a"(dk[dt][1]), "+a"(dv[dt][0]), "+a"(dv[dt][1])::"memory");

    // ---- lane (key, g) holds columns 8 q + 4 g + {0..3}: a swap of the upper half of the one with the lower half of the next
    // makes them 16 bytes of a row
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const int key = nw0 + 32 * b + (lane & 31);
        const bool hidden = PER_KEY && (key >= Nk || (key_mask != nullptr && key_mask[(size_t)(bh / hkv) * N + min(key, N - 1)] == 0));
        const size_t row = head_off + (size_t)key * D + 8 * (lane >> 5);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float mul = i ? scale : 1.0f;
#pragma unroll
            for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
                for (int x = 0; x < 16; x += 8) {
                    const f32x16& a = i ? dk[dt][b] : dv[dt][b];
                    u32x4 v;
#pragma unroll
                    for (int y = 0; y < 2; ++y) {
                        const u32x2 z = __builtin_amdgcn_permlane32_swap(pack_bf16(a[x + 2 * y] * mul, a[x + 2 * y + 1] * mul),
                                                                         pack_bf16(a[x + 4 + 2 * y] * mul, a[x + 5 + 2 * y] * mul), false, false);
                        v[y] = hidden ? 0u : z.x;
                        v[2 + y] = hidden ? 0u : z.y;
                    }
                    if (key < N) st_global_16((i ? dK : dV) + row + 32 * dt + 2 * x, v);
                }
        }
    }
    wait_vmcnt0();                                   // the requests past the end write LDS, which is the next workgroup's then
}

// dK and dV of 64 keys for small launches: waves w and w + 2 own the same 32 keys, one the first and one the second 32 rows of
// every query tile, and exchange at the end (one finishes dV, the other dK).  Half the work a step and twice the workgroups of
// bwd_dkv.  The query tiles of all G heads are one run of steps, three requested ahead into a ring of four stages; the pairs
// of all of them are made first and stay in LDS, so nothing is written that another workgroup reads.  Bound by latencies: a
// step is 32 products of 32 cycles a wave and takes 1.6 us (1.0 at D = 64), of which the pairs are a third.  Tried: one
// product, then its share of the other instructions by scheduling groups (4 % slower), pairs a step ahead instead of first (as slow).
// Not causal with lengths, six registers too many at D = 128 (28 bytes a lane in scratch memory).
template <int D, bool CAUSAL, AttnMask MASK>
__device__ __forceinline__ void bwd_dkv_half(int block,
    const uint16_t* __restrict__ Q, const uint16_t* __restrict__ Kp, const uint16_t* __restrict__ Vp,
    const uint16_t* __restrict__ O, const uint16_t* __restrict__ dO, const float* __restrict__ LSE,
    uint16_t* __restrict__ dK, uint16_t* __restrict__ dV, int BHkv, int N, float scale, float scale_log2, int Hq, int G, int window, const int* __restrict__ kv_lens, const uint8_t* __restrict__ key_mask) {
    using namespace fab;
    using C = CfgK<D>;
    constexpr bool WINDOW = MASK == AttnMask::Limits, PER_KEY = MASK != AttnMask::None;
    constexpr int BNK = 64, STAGE = 2 * C::TILE;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int t = threadIdx.x;
    const int lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int r = lane & 31, g = lane >> 5, T = w >> 1;

    int bh, kt;                           // causal: key tile 0 meets every query tile, so heavy first
    if ((BHkv & 7) == 0) {
        const int slot = block >> 3, heads = BHkv >> 3;
        bh = slot % heads * 8 + (block & 7);
        kt = slot / heads;
    } else {
        bh = block % BHkv;
        kt = block / BHkv;
    }
    const int n0 = kt * BNK, nw0 = n0 + (w & 1) * 32, kvpos = nw0 + r;
    const size_t head_off = (size_t)bh * N * D;
    const int hkv = Hq / G;
    const size_t qh0 = (size_t)(bh / hkv) * Hq + (size_t)(bh % hkv) * G;
    const int Nk = (PER_KEY && kv_lens != nullptr) ? max(0, min(N, kv_lens[bh / hkv])) : N;
    bool block_hidden = PER_KEY && n0 >= Nk;
    if (PER_KEY && key_mask != nullptr && !block_hidden) {
        const TileSpan span = visible_tiles(key_mask + (size_t)(bh / hkv) * N + n0, min(BNK, Nk - n0), lane);
        block_hidden = span.first >= span.last;
    }
    // query tiles [jq0, jq1) of each head see keys of the block
    const int nq = (N + C::BQ - 1) / C::BQ, jq0 = CAUSAL ? kt : 0;
    int jq1 = nq;
    if (WINDOW && window > 0) jq1 = (int)min((int64_t)nq, ((int64_t)n0 + BNK - 2 + window) / C::BQ + 1);
    const int per_head = jq1 - jq0, steps = block_hidden ? 0 : G * per_head;

    const uint32_t head_bytes = (uint32_t)N * D * 2u;
    const u32x4 q_rsrc = make_raw_rsrc(Q + qh0 * N * D, head_bytes * (uint32_t)G);
    const u32x4 do_rsrc = make_raw_rsrc(dO + qh0 * N * D, head_bytes * (uint32_t)G);
    constexpr int ROWS_PER_INST = 1024 / C::ROW;
    int g_voff[C::PT];
#pragma unroll
    for (int m = 0; m < C::PT; ++m) {
        const int row = (w * C::PT + m) * ROWS_PER_INST + lane / C::KCH;
        g_voff[m] = row * C::ROW + swz<D>(row, lane % C::KCH) * 16 - 1024 * m;   // request m carries 1024 m as its immediate offset
    }
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
    const uint32_t wave_dst = __builtin_amdgcn_readfirstlane(lds_base + (uint32_t)w * C::PT * 1024u);
    // steps past the last one are requested beyond the buffers (zeros, no traffic)
    struct Place { int hq, jq; };                    // of a step: its head, its query tile
    auto next = [&](Place& p) {
        if (++p.jq == jq1) { p.jq = jq0; ++p.hq; }
    };
    auto issue_rows = [&](int at, const Place& p) {
        const uint32_t dst = wave_dst + (uint32_t)(at & (C::NST - 1)) * STAGE;
        const int soff = at < steps ? p.hq * (int)head_bytes + p.jq * C::BQ * C::ROW : (int)(head_bytes * (uint32_t)G);
        load_global_to_lds_16xN<C::PT>(q_rsrc, dst, g_voff, soff);
        load_global_to_lds_16xN<C::PT>(do_rsrc, dst + C::TILE, g_voff, soff);
    };
    Place ahead{0, jq0};                             // of the next step to request
#pragma unroll
    for (int at = 0; at < 3; ++at) {
        issue_rows(at, ahead);
        next(ahead);
    }
    bf16x8 kf[C::KSTEPS], vf[C::KSTEPS];
    {
        const size_t off = head_off + (size_t)min(kvpos, N - 1) * D + g * 8;
#pragma unroll
        for (int i = 0; i < C::KSTEPS; ++i) {
            kf[i] = __builtin_bit_cast(bf16x8, ld_global_16(Kp + off + i * 16));
            vf[i] = __builtin_bit_cast(bf16x8, ld_global_16(Vp + off + i * 16));
        }
    }
    // The (lse2, delta = dO . O) pairs of all steps, in LDS behind the stages.  A row is 16 bytes a lane of D / 8 adjacent lanes and
    // the loads of four tiles are in flight.  (A row a lane, as the products want them, and through memory, as bwd_dkv makes them:
    // 1 us a tile, as much as its step.)
    float2* pairs = reinterpret_cast<float2*>(lds + C::NST * STAGE);
    {
        constexpr int LPR = D / 8, ROWS = THREADS / LPR, PASSES = C::BQ / ROWS, TILES = 4;
        const int row = t / LPR, c = t % LPR;
        Place p{0, jq0};
        for (int s0 = 0; s0 < steps; s0 += TILES) {
            u32x4 o[TILES][PASSES], d[TILES][PASSES];
            float lse[TILES][PASSES];
            int qpos[TILES];
#pragma unroll
            for (int i = 0; i < TILES; ++i)
                if (s0 + i < steps) {
                    qpos[i] = p.jq * C::BQ + row;
#pragma unroll
                    for (int k = 0; k < PASSES; ++k) {
                        const size_t at = (qh0 + p.hq) * N + min(qpos[i] + k * ROWS, N - 1);
                        o[i][k] = ld_global_16(O + at * D + c * 8);
                        d[i][k] = ld_global_16(dO + at * D + c * 8);
                        lse[i][k] = LSE[at];
                    }
                    next(p);
                }
#pragma unroll
            for (int i = 0; i < TILES; ++i)
                if (s0 + i < steps) {
#pragma unroll
                    for (int k = 0; k < PASSES; ++k) {
                        float delta = dot8_bf16(d[i][k], o[i][k]);
                        // lanes xor 1, xor 2, then the mirrored half row and row: sums of 4, 8 and 16 lanes
                        auto add = [&](auto ctrl) {
                            delta += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, delta), decltype(ctrl)::value, 0xf, 0xf, true));
                        };
                        add(std::integral_constant<int, 0xb1>{});
                        add(std::integral_constant<int, 0x4e>{});
                        add(std::integral_constant<int, 0x141>{});
                        if (LPR == 16) add(std::integral_constant<int, 0x140>{});
                        float lse2 = lse[i][k] * LOG2E;
                        if (MASK != AttnMask::None && lse2 == -INFINITY) lse2 = INFINITY;    // a row that saw no key: every probability is 0
                        if (c == 0) pairs[(s0 + i) * C::BQ + row + k * ROWS] = qpos[i] + k * ROWS < N ? make_float2(lse2, delta) : make_float2(INFINITY, 0.0f);
                    }
                }
        }
    }
    Place now{0, jq0};
#pragma unroll
    for (int i = 0; i < C::KSTEPS; ++i) { pin_registers(kf[i]); pin_registers(vf[i]); }
    wait_vmcnt0();
    __syncthreads();

    // fragment addresses inside a stage, of this wave's 32 rows
    int row_off[C::KSTEPS], tr_lo[C::DT], tr_hi[C::DT];
#pragma unroll
    for (int i = 0; i < C::KSTEPS; ++i) row_off[i] = (32 * T + r) * C::ROW + swz<D>(r, 2 * i + g) * 16;
    {
        const int i16 = lane & 15, b16 = lane >> 4, row = 4 * (b16 >> 1) + (i16 >> 2);
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt) {
            const int dcol = 32 * dt + 16 * (b16 & 1) + 4 * (i16 & 3);
            tr_lo[dt] = (32 * T + row) * C::ROW + swz<D>(row, dcol >> 3) * 16 + (dcol & 7) * 2;
            tr_hi[dt] = (32 * T + row + 8) * C::ROW + swz<D>(row + 8, dcol >> 3) * 16 + (dcol & 7) * 2;
        }
    }
    f32x16 dk[C::DT], dv[C::DT];
#pragma unroll
    for (int i = 0; i < C::DT; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) { dk[i][e] = 0.0f; dv[i][e] = 0.0f; }

    auto scores = [&](int at, f32x16& s, f32x16& dp) {
        const unsigned char* St = lds + (at & (C::NST - 1)) * STAGE;
        bf16x8 qa[C::KSTEPS], da[C::KSTEPS];
#pragma unroll
        for (int i = 0; i < C::KSTEPS; ++i) {
            qa[i] = *reinterpret_cast<const bf16x8*>(St + row_off[i]);
            da[i] = *reinterpret_cast<const bf16x8*>(St + C::TILE + row_off[i]);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] = dp[e] = 0.0f;
#pragma unroll
        for (int i = 0; i < C::KSTEPS; ++i) {
            s = mfma_32x32x16_bf16(qa[i], kf[i], s);
            dp = mfma_32x32x16_bf16(da[i], vf[i], dp);
        }
    };
    // The products of the next step's scores stand beside this step's exponentials: tile at + 1 is awaited a step early.
    auto step = [&](int at, const f32x16& s, const f32x16& dp, f32x16& s_next, f32x16& dp_next) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * C::PT) : "memory");
        __syncthreads();
        issue_rows(at + 3, ahead);                   // into the stage of the step before
        next(ahead);
        const int qs0 = now.jq * C::BQ + 32 * T;
        next(now);
        const unsigned char* St = lds + (at & (C::NST - 1)) * STAGE;
        // register e of a product <-> query row qs0 + 8 (e / 4) + 4 g + e % 4
        f32x4 pair[8];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float2* p = pairs + at * C::BQ + 32 * T + 4 * g + 8 * k;
            pair[2 * k] = *reinterpret_cast<const f32x4*>(p);
            pair[2 * k + 1] = *reinterpret_cast<const f32x4*>(p + 2);
        }
        scores(at + 1, s_next, dp_next);
        bf16x8 dot[2][C::DT], qt[2][C::DT];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int dt = 0; dt < C::DT; ++dt) {
                const unsigned char* lo = St + tr_lo[dt] + c * 16 * C::ROW;
                const unsigned char* hi = St + tr_hi[dt] + c * 16 * C::ROW;
                dot[c][dt] = __builtin_shufflevector(ds_read_tr16(lo + C::TILE), ds_read_tr16(hi + C::TILE), 0, 1, 2, 3, 4, 5, 6, 7);
                qt[c][dt] = __builtin_shufflevector(ds_read_tr16(lo), ds_read_tr16(hi), 0, 1, 2, 3, 4, 5, 6, 7);
            }
        // selected, not branched over: a branch would end the block that the products and this are interleaved in
        const int row_lo = CAUSAL && qs0 < nw0 + 32 ? kvpos - qs0 - 4 * g : INT_MIN;                 // rows below are hidden
        const int row_hi = WINDOW && window > 0 && qs0 + 31 - nw0 >= window ? kvpos + window - qs0 - 4 * g : INT_MAX;       // and from here on
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            u32x4 ppk, dpk;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int k = 2 * c + h;
                float p[4], ds[4];
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    p[x] = fast_exp2(fmaf(s[4 * k + x], scale_log2, -pair[2 * k + x / 2][2 * (x & 1)]));
                    if (CAUSAL) p[x] = 8 * k + x < row_lo ? 0.0f : p[x];
                    if (WINDOW) p[x] = 8 * k + x >= row_hi ? 0.0f : p[x];
                    ds[x] = p[x] * (dp[4 * k + x] - pair[2 * k + x / 2][2 * (x & 1) + 1]);
                }
                ppk[2 * h] = pack_bf16(p[0], p[1]);
                ppk[2 * h + 1] = pack_bf16(p[2], p[3]);
                dpk[2 * h] = pack_bf16(ds[0], ds[1]);
                dpk[2 * h + 1] = pack_bf16(ds[2], ds[3]);
            }
            const bf16x8 pf = __builtin_bit_cast(bf16x8, ppk), dsf = __builtin_bit_cast(bf16x8, dpk);
#pragma unroll
            for (int dt = 0; dt < C::DT; ++dt) {
                dv[dt] = mfma_32x32x16_bf16(dot[c][dt], pf, dv[dt]);
                dk[dt] = mfma_32x32x16_bf16(qt[c][dt], dsf, dk[dt]);
            }
        }
    };
    f32x16 sA, dpA, sB, dpB;
    if (steps > 0) scores(0, sA, dpA);
    for (int at = 0; at < steps; at += 2) {
        step(at, sA, dpA, sB, dpB);
        if (at + 1 < steps) step(at + 1, sB, dpB, sA, dpA);
    }
    wait_vmcnt0();
    __syncthreads();                                 // the stages are free
    if constexpr (PER_KEY) {
        if (kvpos >= Nk || (key_mask != nullptr && key_mask[(size_t)(bh / hkv) * N + min(kvpos, N - 1)] == 0)) {
#pragma unroll
            for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
                for (int e = 0; e < 16; ++e) dv[dt][e] = dk[dt][e] = 0.0f;
        }
    }
    // waves 0, 1 give dK away and finish dV, waves 2, 3 the other way round
    f32x4* give = reinterpret_cast<f32x4*>(lds) + w * (C::DT * 4 * 64) + lane;
    const f32x4* take = reinterpret_cast<const f32x4*>(lds) + (w ^ 2) * (C::DT * 4 * 64) + lane;
    unsigned char* scratch = lds + 4 * C::DT * 4 * 64 * 16 + w * (32 * (D * 2 + 16));
    static_assert(4 * C::DT * 4 * 64 * 16 + 4 * 32 * (D * 2 + 16) <= C::NST * STAGE, "exchange and transposition");
    auto hand_over = [&](const f32x16 (&v)[C::DT]) {
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) give[(dt * 4 + q4) * 64] = f32x4{v[dt][4 * q4], v[dt][4 * q4 + 1], v[dt][4 * q4 + 2], v[dt][4 * q4 + 3]};
    };
    auto finish = [&](f32x16 (&v)[C::DT], float mul, uint16_t* out) {
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                const f32x4 other = take[(dt * 4 + q4) * 64];
#pragma unroll
                for (int x = 0; x < 4; ++x) v[dt][4 * q4 + x] += other[x];
            }
        store_transposed_bf16<D>(v, mul, scratch, out + head_off + (size_t)nw0 * D, N - nw0, lane);
    };
    if (T == 0) hand_over(dk); else hand_over(dv);
    __syncthreads();
    if (T == 0) finish(dv, 1.0f, dV); else finish(dk, scale, dK);
}

// Both at once for launches that leave CUs idle anyway (launch_us): the first `ndkv` workgroups are dK/dV's, the
// rest dQ's (64-row form).  HALF: dK/dV by bwd_dkv_half.
// The dQ kernel then need not end before dK/dV starts -- a launch, a prologue and a drain, 3.5 us of 11 for one head of 128 rows,
// 12 of 41 for 8 heads of 700.
template <int D, bool CAUSAL, AttnMask MASK, bool CUT, bool HALF>
__global__ __launch_bounds__(fab::THREADS, D == 64 && HALF ? 2 : 1) void flash_attn_bwd_both_kernel(
    const uint16_t* __restrict__ Q, const uint16_t* __restrict__ Kp, const uint16_t* __restrict__ Vp,
    const uint16_t* __restrict__ O, const uint16_t* __restrict__ dO, const float* __restrict__ LSE,
    uint16_t* __restrict__ dQ, float2* stats, uint16_t* __restrict__ dK, uint16_t* __restrict__ dV, int BH, int N, int ntq,
    int ntk, int npad, float scale, float scale_log2, int Hq, int window, const int* __restrict__ kv_lens,
    const uint8_t* __restrict__ key_mask, int single, fab::Parts plan, int items, float* __restrict__ partial, int ndkv) {
    const int at = blockIdx.x;
    if (HALF && at < ndkv) {
        bwd_dkv_half<D, CAUSAL, MASK>(at, Q, Kp, Vp, O, dO, LSE, dK, dV, BH / plan.G, N, scale, scale_log2, Hq, plan.G,
                                      window, kv_lens, key_mask);
    } else if (at < ndkv) {
        bwd_dkv<D, CAUSAL, MASK, CUT, true, false>(at, Q, Kp, Vp, O, dO, LSE, stats, dK, dV, BH / plan.G, N, ntk, npad, scale, scale_log2, Hq,
                                         window, kv_lens, key_mask, plan, items, partial, nullptr);
    } else {
        bwd_dq<D, CAUSAL, MASK, true>(at - ndkv, Q, Kp, Vp, O, dO, LSE, dQ, nullptr, BH, N, ntq, npad, scale, scale_log2, Hq, plan.G,
                                      window, kv_lens, key_mask, 0, single, 0);
    }
}

// ------------------------------------------------------------------------------------------
// (lse * log2 e, delta) of every query row for dK/dV launches that no dQ launch precedes: delta = dO . O, rows of the padding
// up to npad get (+inf, 0).  16 bytes a lane of each operand; bound by HBM.
template <int D>
__global__ __launch_bounds__(256) void flash_attn_bwd_stats_kernel(const uint16_t* __restrict__ O, const uint16_t* __restrict__ dO,
                                                                  const float* __restrict__ LSE, float2* __restrict__ stats, int N,
                                                                  int npad, int masked) {
    constexpr int LANES = D / 8, ROWS = 256 / LANES;
    const int per_head = npad / ROWS;
    const int bh = blockIdx.x / per_head, qpos = blockIdx.x % per_head * ROWS + threadIdx.x / LANES, qrow = min(qpos, N - 1);
    const size_t off = ((size_t)bh * N + qrow) * D + threadIdx.x % LANES * 8;
    float delta = fab::dot8_bf16(ld_global_16(dO + off), ld_global_16(O + off));
    float lse2 = LSE[(size_t)bh * N + qrow] * fab::LOG2E;
#pragma unroll
    for (int x = 1; x < LANES; x <<= 1) delta += __shfl_xor(delta, x, 64);
    if (masked && lse2 == -INFINITY) lse2 = INFINITY;                // a row that saw no key: every probability is 0
    if (threadIdx.x % LANES == 0) stats[(size_t)bh * npad + qpos] = qpos < N ? make_float2(lse2, delta) : make_float2(INFINITY, 0.0f);
}

// dQ = dS K of the dS that the dK/dV launch left: one workgroup = 128 query rows (4 waves x 32), a ring of stages of 32 keys
// (four 2 KB blocks of dS, 32 rows of K) filled by global -> LDS requests, products transposed as in flash_attn_bwd_dq_kernel:
//    dQ^T (D x 32 q) += K_tile^T x dS^T
// both operands by transposing reads.  Bound by the L2 -> LDS requests (B1 Hq32 Hkv8 N2000: 29 us for 142 MB of dS and as much of K; without
// its products the kernel takes as long).  256 rows a workgroup halve the K part and take 36 us there: the longest has a CU to
// itself.  Fragments read ahead of their products, across the stages: 30 us.
namespace fab {
template <int D>
struct CfgP {
    static constexpr int BM = 128, BN = 32, NST = 5; // two workgroups a CU share its 160 KB
    static constexpr int ROW = D * 2, KCH = D / 8;
    static constexpr int DS = 4 * 2048, STAGE = DS + BN * ROW, LDS = NST * STAGE;
    static constexpr int PT = BN * KCH / THREADS;    // 16-byte chunks of K per thread and stage
    static constexpr int LOADS = 2 + PT, DT = D / 32;
};
}  // namespace fab
template <int D, bool CAUSAL, AttnMask MASK>
__device__ __forceinline__ void bwd_dq_product(int block, const uint16_t* __restrict__ Kp, const unsigned char* __restrict__ ds,
                                               uint16_t* __restrict__ dQ, int BH, int N, int ntq, float scale, int Hq, int G,
                                               int window, const int* __restrict__ kv_lens, const uint8_t* __restrict__ key_mask,
                                               int single) {
    using namespace fab;
    using C = CfgP<D>;
    constexpr bool LIMITS = MASK == AttnMask::Limits, KEYS = MASK == AttnMask::Keys;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int t = threadIdx.x;
    const int lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);

    int bh, rank, kvbh;
    AttnOrder{BH, Hq, G, ntq, single}.decode(block, bh, rank, kvbh);
    const int qt = CAUSAL ? ntq - 1 - rank : rank;
    const int q0 = qt * C::BM, qw0 = q0 + w * 32;
    const int Nk = (LIMITS && kv_lens != nullptr) ? max(0, min(N, kv_lens[bh / Hq])) : N;
    int kv_end = CAUSAL ? min(Nk, q0 + C::BM) : Nk;
    int begin = (LIMITS && window > 0) ? max(0, q0 - window + 1) / C::BN : 0;      // stages = 32 keys
    if constexpr (KEYS) {
        const TileSpan span = visible_tiles(key_mask + (size_t)(bh / Hq) * N, kv_end, lane);
        begin = 2 * span.first;
        kv_end = min(kv_end, 64 * span.last);
    }
    const int end = (kv_end + C::BN - 1) / C::BN;
    // the stages that hold a visible pair for this wave's rows: only those blocks are written for certain
    const int wave_end = CAUSAL ? min(end, qw0 / C::BN + 1) : end;
    const int wave_begin = (LIMITS && window > 0) ? max(0, qw0 - window + 1) / C::BN : begin;

    const DsBlocks place{ntq, CAUSAL, LIMITS ? window : 0};
    const int tile_bytes = place.tiles(qt) * 16 * 2048, s_first = 4 * place.first(qt);
    const u32x4 s_rsrc = make_raw_rsrc(ds + (size_t)bh * place.head_bytes() + place.at(qt) * 2048, (uint32_t)tile_bytes);
    const u32x4 k_rsrc = make_raw_rsrc(Kp + (size_t)kvbh * N * D, (uint32_t)N * D * 2u);
    constexpr int ROWS_PER_INST = 1024 / C::ROW;
    int s_voff[2], k_voff[C::PT];                    // request m carries 1024 m as its immediate offset
    s_voff[0] = s_voff[1] = w * 2048 + lane * 16;
#pragma unroll
    for (int m = 0; m < C::PT; ++m) {
        const int row = (w * C::PT + m) * ROWS_PER_INST + lane / C::KCH;
        k_voff[m] = row * C::ROW + swz<D>(row, lane % C::KCH) * 16 - 1024 * m;
    }
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
    const uint32_t s_dst = __builtin_amdgcn_readfirstlane(lds_base + (uint32_t)w * 2048u);
    const uint32_t k_dst = __builtin_amdgcn_readfirstlane(lds_base + C::DS + (uint32_t)w * C::PT * 1024u);
    // stages past the end are requested beyond the buffers (zeros, no traffic), so that the wait count below is constant
    auto issue = [&](uint32_t at, int j) {
        load_global_to_lds_16xN<2>(s_rsrc, s_dst + at, s_voff, j < end ? (j - s_first) * C::DS : tile_bytes);
        load_global_to_lds_16xN<C::PT>(k_rsrc, k_dst + at, k_voff, j < end ? j * C::BN * C::ROW : N * C::ROW);
    };
    // transposing reads: keys 16 c + 4 (lane / 32) + {0..3} and 8 more, in the same order of both operands
    int tr_lo[C::DT], tr_hi[C::DT], s_lo, s_hi;
    {
        const int i16 = lane & 15, b16 = lane >> 4, row = 4 * (b16 >> 1) + (i16 >> 2);
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt) {
            const int dcol = 32 * dt + 16 * (b16 & 1) + 4 * (i16 & 3);
            tr_lo[dt] = C::DS + row * C::ROW + swz<D>(row, dcol >> 3) * 16 + (dcol & 7) * 2;
            tr_hi[dt] = C::DS + (row + 8) * C::ROW + swz<D>(row + 8, dcol >> 3) * 16 + (dcol & 7) * 2;
        }
        // dS pieces as store_ds deals them: half sh = b16 & 1, its g = lane & 1, rows + 8 in the upper 8 bytes
        const int sh = b16 & 1, gp = i16 & 1, x = 4 * gp + 8 * sh;
        s_lo = w * 2048 + sh * 1024 + (gp * 32 + (row ^ x)) * 16 + ((i16 >> 1) & 1) * 8;
        s_hi = w * 2048 + sh * 1024 + (gp * 32 + ((row + 8) ^ x)) * 16 + ((i16 >> 1) & 1) * 8;
    }
    f32x16 dq[C::DT];
#pragma unroll
    for (int i = 0; i < C::DT; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) dq[i][e] = 0.0f;

#pragma unroll
    for (int i = 0; i < C::NST - 1; ++i) issue(i * C::STAGE, begin + i);
    uint32_t at = 0;                                 // the stage's place in the ring
    for (int j = begin; j < end; ++j) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((C::NST - 2) * C::LOADS) : "memory");
        __syncthreads();                             // stage j is here; the one before it has been read by every wave
        issue(at == 0 ? (C::NST - 1) * C::STAGE : at - C::STAGE, j + C::NST - 1);
        if (j >= wave_begin && j < wave_end) {
            const unsigned char* St = lds + at;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const bf16x4 dl = ds_read_tr16(St + s_lo + c * 256), dh = ds_read_tr16(St + s_hi + c * 256);
                const bf16x8 dsf = __builtin_shufflevector(dl, dh, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                for (int dt = 0; dt < C::DT; ++dt) {
                    const bf16x4 lo = ds_read_tr16(St + tr_lo[dt] + c * 16 * C::ROW), hi = ds_read_tr16(St + tr_hi[dt] + c * 16 * C::ROW);
                    dq[dt] = mfma_32x32x16_bf16(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), dsf, dq[dt]);
                }
            }
        }
        at = at == (C::NST - 1) * C::STAGE ? 0 : at + C::STAGE;
    }
    wait_vmcnt0();
    __syncthreads();
    store_transposed_bf16<D>(dq, scale, lds + w * (32 * (D * 2 + 16)), dQ + ((size_t)bh * N + qw0) * D, N - qw0, lane);
}

// dK and dV of the key tiles that were cut into parts: the parts' f32 sums added in order, 8 elements of a row per thread.
template <int D>
__device__ __forceinline__ void bwd_sum(int block, const float* __restrict__ partial, uint16_t* __restrict__ dK,
                                        uint16_t* __restrict__ dV, int N, int ntk, int items, float scale, fab::Parts plan) {
    constexpr int CH = D / 8, DT = D / 32, TILE16 = 2 * 4 * DT * 4 * 64;      // 16-byte pieces of one part
    const int id = block * 256 + threadIdx.x;
    constexpr int PER_TILE = 2 * 128 * CH;
    const int tile = (block * 256) / PER_TILE;                          // a workgroup stays inside one tile
    const int bh = tile / ntk, kt = tile % ntk;
    const int parts = plan.parts(kt);
    if (parts == 1) return;
    int first = 0;
    for (int k = 0; k < kt; ++k) first += plan.parts(k);
    const int within = id % PER_TILE, which = within / (128 * CH), row = (within / CH) % 128, c = within % CH;
    // d = 8c .. 8c + 7 of key row `row`: register group dt = c / 4, q4 = c % 4 of wave row / 32, lanes row % 32 (+ 32)
    const f32x4* in = reinterpret_cast<const f32x4*>(partial) + ((size_t)bh * items + first) * TILE16 +
                      (which * 4 * DT * 4 + (row >> 5) * (DT * 4) + c) * 64 + (row & 31);
    f32x4 lo = in[0], hi = in[32];
    for (int p = 1; p < parts; ++p) {
        lo += in[(size_t)p * TILE16];
        hi += in[(size_t)p * TILE16 + 32];
    }
    if (kt * 128 + row >= N) return;
    const float mul = which ? scale : 1.0f;
    u32x4 v;
    v[0] = pack_bf16(lo[0] * mul, lo[1] * mul);
    v[1] = pack_bf16(lo[2] * mul, lo[3] * mul);
    v[2] = pack_bf16(hi[0] * mul, hi[1] * mul);
    v[3] = pack_bf16(hi[2] * mul, hi[3] * mul);
    st_global_16((which ? dK : dV) + ((size_t)bh * N + kt * 128 + row) * D + c * 8, v);
}

template <int D>
__global__ __launch_bounds__(256) void flash_attn_bwd_sum_kernel(const float* __restrict__ partial, uint16_t* __restrict__ dK,
                                                                uint16_t* __restrict__ dV, int N, int ntk, int items, float scale,
                                                                fab::Parts plan) {
    bwd_sum<D>(blockIdx.x, partial, dK, dV, N, ntk, items, scale, plan);
}
// The launch after a dK/dV launch that left dS: the first `ndq` workgroups are dQ's, the rest add the parts, on the CUs that
// short dQ tiles leave (B1 Hq32 Hkv8 N2000: 28 + 8 us in two launches).
template <int D, bool CAUSAL, AttnMask MASK>
__global__ __launch_bounds__(fab::THREADS, 2) void flash_attn_bwd_dq_product_kernel(
    const uint16_t* __restrict__ Kp, const unsigned char* __restrict__ ds, uint16_t* __restrict__ dQ, int BH, int N, int ntq,
    float scale, int Hq, int window, const int* __restrict__ kv_lens, const uint8_t* __restrict__ key_mask, int single, int ndq,
    const float* __restrict__ partial, uint16_t* __restrict__ dK, uint16_t* __restrict__ dV, int items, fab::Parts plan) {
    const int at = blockIdx.x;
    if (at < ndq) bwd_dq_product<D, CAUSAL, MASK>(at, Kp, ds, dQ, BH, N, ntq, scale, Hq, plan.G, window, kv_lens, key_mask, single);
    else bwd_sum<D>(at - ndq, partial, dK, dV, N, ntq, items, scale, plan);
}

size_t flash_attn_bwd_workspace_bytes(int B, int H, int N) {
    const size_t npad = ((size_t)N + 127) / 128 * 128;
    return (size_t)B * H * npad * sizeof(float2);
}

namespace {
// One of the eight XCDs, which are alike: it gets every eighth workgroup of a launch and deals them to its four engines of eight CUs
// in turn; the next one waits until the engine whose turn it is has a free place (fab::Parts::order).
struct Xcd {
    int places;                                      // of an engine: 8, or 16 where two workgroups share a CU
    double free_at[4][16] = {}, started = 0, last = 0;
    int n = 0;
    void run(double us) {
        double* at = std::min_element(free_at[n & 3], free_at[n & 3] + places);
        ++n;
        started = std::max(started, *at);
        *at = started + us;
        last = std::max(last, *at);
    }
};
// The steps of the dK / dV workgroups that go to the first XCD, in the launch's order (bwd_dkv).
template <class F> void first_xcd_dkv(const fab::Parts& p, int ntk, int BHkv, F&& run) {
    const bool xcds = BHkv % 8 == 0;
    const int heads = xcds ? BHkv / 8 : BHkv, stride = xcds ? 1 : 8;
    if (p.chunk) {
        for (int kt = 0, at = 0; kt < ntk; ++kt)
            for (const int end = at + p.parts(kt) * heads; at < end; ++at)
                if (at % stride == 0) run(p.part_steps(kt));
    } else {
        for (int at = 0; at < heads * ntk; at += stride) {
            int kt;
            p.order(at, heads, xcds, ntk, kt);
            run(p.steps(kt));
        }
    }
}
// When the last CU is done, with workgroups of wg + step * steps
double last_cu(const fab::Parts& p, int ntk, int BHkv, double wg, double step) {
    Xcd x{8};
    first_xcd_dkv(p, ntk, BHkv, [&](int steps) { x.run(wg + step * steps); });
    return x.last;
}
// traffic of the f32 partials, written and read at 6 TB/s
double partial_us(const fab::Parts& p, int BHkv, int N, int D) {
    int64_t cut = 0;
    for (int kt = 0; kt < (N + 127) / 128; ++kt) cut += p.parts(kt) > 1 ? p.parts(kt) : 0;
    return cut * BHkv * (128.0 * D * 8 * 2) / 6.0e6;
}
// How the dK / dV work is cut.  A workgroup has a CU to itself.  A step (64 queries x 128 keys) takes 1.7 us at D = 128 (1.1
// at 64) while other CUs are idle and a quarter more with all of them busy (measured: 1.65-1.75 with the last key tiles of
// a head alone on the device, 2.0-2.2 with 256 equal workgroups, 1.95 in the large launches), a workgroup 2 us to start and
// end, the sum of the parts 3 us and the traffic of its partials (written and read at 6 TB/s).  Tried: whole key tiles, and
// the finest cut with at most 256, 512 or 768 workgroups.  On 235 shapes (1 to 16 sequences of 64 to 8192 rows, every mask)
// the choice is 0.2 % slower than the best of the four, at worst 11 % (B6 Hq32 Hkv8 N92).  With 1.55 us for every step and
// whole tiles taken longest first it was 1.7 %, at worst 45 %: B9 Hq16 Hkv4 N1944 ran whole, 832 us for 573 in parts.
struct DkvPlan {
    fab::Parts parts;
    double us;
};
DkvPlan make_dkv_plan(int BHkv, int G, int N, int D, bool causal, int window, bool cut_tiles) {
    const int ntk = (N + 127) / 128, nq = (N + 63) / 64;
    const fab::Parts whole{G, nq, causal, window, 0, 128};
    DkvPlan best{whole, 1e300};
    const double step = D == 128 ? 1.7 : 1.1;
    int64_t total = 0;
    int most = 1;
    for (int kt = 0; kt < ntk; ++kt) {
        total += whole.steps(kt);
        most = std::max(most, whole.steps(kt));
    }
    const double mean = (double)total * BHkv / 256;           // steps of a CU if all were equally busy
    const bool few = ntk <= 64 && (int64_t)ntk * BHkv <= 768;
    for (int round = 0; round <= (cut_tiles && few ? 3 : 0); ++round) {
        fab::Parts p = whole;
        auto count = [&](int chunk) {
            p.chunk = chunk;
            int64_t n = 0;
            for (int kt = 0; kt < ntk; ++kt) n += p.parts(kt);
            return n * BHkv;
        };
        int64_t n = (int64_t)ntk * BHkv, cut = 0;
        if (round) {
            int lo = std::max<int64_t>(2, total * BHkv / (256 * round)), hi = most;     // least chunk with few enough parts
            if (lo >= hi || count(hi) > 256 * round) continue;
            while (lo < hi) {
                const int mid = (lo + hi) / 2;
                if (count(mid) <= 256 * round) hi = mid; else lo = mid + 1;
            }
            n = count(lo);
            for (int kt = 0; kt < ntk; ++kt) cut += p.parts(kt) > 1 ? p.parts(kt) : 0;
            if (cut == 0) continue;
        }
        const double last = n <= 2048 ? last_cu(p, ntk, BHkv, 0, 1) : mean + 0.5 * most;
        double us = step * std::max(last, 1.25 * mean) + 2.0 * std::max(1.0, n / 256.0);
        if (round) us += 3.0 + partial_us(p, BHkv, N, D);
        // A tie goes to the parts at D = 128 where an XCD has several heads.  It decides 62 of 8000 shapes, which take the same time in the
        // mean with this and without, 0.91 to 1.14 times one by one (B3 Hq16 Hkv4 N4054 with a key mask 545 us and 623, B2 Hq32 Hkv8 N4158 797
        // and 726).
        if (us < best.us * (best.parts.chunk == 0 && D == 128 && BHkv > 8 ? 1.045 : 1.0)) best = {p, us};
    }
    return best;
}
// What key tiles of 256 save a dQ launch and a dK/dV launch one after the other: a workgroup of them takes 13.5 us and 2.3 a step (64
// queries x 256 keys) at D = 128, 8.3 and 1.6 at 64, in a launch that fills the device; plan.us against that, as the two were measured.
// On 556 shapes (1 to 16 sequences of 64 to 8192 rows, 1 to 32 heads, every mask) the choice is 0.1 % slower than the better of the two
// at D = 128 and 0.3 % at 64; there are 117 shapes where the wide tiles are the faster ones, by up to 23 %.
double wide_saves(int BHkv, int G, int N, int D, bool causal, int window, const DkvPlan& plan) {
    const int ntk = (N + 255) / 256;
    const fab::Parts wide{G, (N + 63) / 64, causal, window, 0, 256};
    const double wg = D == 128 ? 13.5 : 8.3, step = D == 128 ? 2.29 : 1.59;
    double us;
    if ((int64_t)ntk * BHkv <= 16384) {
        us = last_cu(wide, ntk, BHkv, wg, step);
    } else {
        int64_t steps = 0;
        for (int kt = 0; kt < ntk; ++kt) steps += wide.steps(kt);
        us = (wg * ntk + step * (double)steps) * BHkv / 256;
    }
    return (D == 128 ? 0.89 * plan.us + 8.7 : 0.957 * plan.us + 5.1) - us;
}
int dkv_items(const fab::Parts& p, int N) {
    const int ntk = (N + p.keys - 1) / p.keys;
    if (p.chunk == 0) return ntk;
    int n = 0;
    for (int kt = 0; kt < ntk; ++kt) n += p.parts(kt);
    return n;
}
// At D = 64 two workgroups of 64-key tiles fit a CU, and do where there are more than CUs and all take as long (B1 H16 N514 not causal
// 20.6 -> 16.0 us, B12 H4 N237 window 157 15.7 -> 11.2).  Causal ones are kept apart by the LDS they ask for: the longest must not share
// its CU (B15 Hq16 Hkv4 N64 9.7 us, 10.5 beside others); nor must the dK/dV ones of grouped heads while they have one each (B2 Hq32
// Hkv8 N257 window 79 20.3, 21.3).
bool kept_apart(int G, int N, bool causal, int window, int64_t workgroups) {
    return (causal && (window <= 0 || window > N / 2)) || (G > 1 && workgroups <= 512);
}
size_t half_lds(int D, int steps, bool apart) {
    const size_t bytes = (size_t)4 * 2 * 64 * D * 2 + (size_t)steps * 64 * sizeof(float2);
    return apart ? std::max<size_t>(bytes, 82 * 1024) : bytes;
}
size_t dkv_partial_bytes(const fab::Parts& p, int BHkv, int N, int D) {
    return p.chunk ? (size_t)BHkv * dkv_items(p, N) * 128 * D * 8 : 0;
}
size_t ds_bytes(int BH, int N, bool causal, int window) {
    return (size_t)BH * fab::DsBlocks{(N + 127) / 128, causal, window}.head_bytes();
}
// The four forms of a backward: dQ and dK/dV one after the other (seven products); in one launch; dK/dV leaving dS for dQ (five
// products, three launches); in one launch with 64-key tiles.
enum Form { TWO, ONE, DS, HALF, FORMS };
constexpr size_t kMostDs = (size_t)288 << 20;        // about the 256 MB last-level cache; with 331 MB B5 Hq8 Hkv2 N2724 300 -> 307 us
int half_steps(int G, int N, bool causal, int window) {                 // of the longest 64-key tile
    const int nq = (N + 63) / 64;
    return G * (causal && window > 0 ? (int)std::min<int64_t>(nq, ((int64_t)window + 62) / 64 + 1) : nq);
}
// What each form takes, in microseconds on an MI355X: the workgroups' times (start and end, and a step: 64 queries x 64 or 128 keys)
// dealt to the CUs in the launch's order as an XCD deals them (Xcd), or the estimates that dQ's and dK/dV's own plans are chosen by, weighted as they
// follow one another.  Steps take longer with all CUs busy (`crowd`) and with the mask instructions of a window (`edges`).
// The constants are near what single workgroups measure and are fitted to make the choice, over 3900 shapes (heads 1 to 32, 64 to 8192
// rows, every mask; graphs of 12 calls); a form's estimate is within 8 to 11 %.  On 1000 other small launches the form chosen is 0.3 %
// slower than the best of the four at D = 128 and 0.6 % at 64, at worst 21 % (B13 H16 N159 causal: 46 us with dS, 38 by 256-key tiles) and 17 %.
// Examples, two / one / dS / half:  D = 128 B1 Hq32 Hkv8 N2000 149 / - / 137 / -, B2 H16 N483 full 36 / 28 / 33 / 34, B5 H8 N217 full 25
// / 18 / 22 / 20, B2 H8 N685 40 / 38 / 32 / 27; D = 64 B1 H1 N128 11.4 / 8.3 / - / 6.6, B9 H8 N66 full 11.5 / 8.3 / - / 8.0, B10
// Hq32 Hkv8 N222 full 42 / - / - / 35, B1 H32 N315 full 16.9 / 14.0 / - / 11.3, B1 Hq16 Hkv4 N1042 full 46 / 56 / - / 68, B1 H2 N2001 41 / 31 / - / 37.
struct FormModel {
    double half, half_wg, half_step;                 // launch; dK/dV workgroup and step
    double dq_wg, dq_tile;                           // dQ's 64-row workgroups beside either
    double one, part_wg, part_step, sum, traffic;    // launch; dK/dV; the addition of parts and its partials
    double two, two_dq, two_dkv;
    double crowd, edges;
    double beside;                                   // what a workgroup of HALF takes longer beside a second one on its CU
    double ds, ds_bytes, ds_dkv, ds_tile, ds_mean, ds_sum;      // launches; pairs, per MB of O and dO; dK/dV; product: longest, mean; parts
};
constexpr FormModel kModel128{3.64, 3.15, 1.77, 3.96, 0.86, 0.544, 7.62, 2.26, 3.06, 1.48, 7, 0.687, 1.34, 0.152, 1.2, 0, 11.4, 0.291, 0.913, 0.215, 1.09, 0.074};
constexpr FormModel kModel64{1.46, 3.28, 1.04, 2.79, 0.7, 2, 4.63, 1.83, 2.29, 1.14, 2.46, 1.07, 1.14, 0.0436, 1.13, 0.3, 0, 0, 0, 0, 0, 0};
void launch_us(const FormModel& m, int BH, int BHkv, int N, int D, bool causal, int window, const DkvPlan& plan, double (&us)[FORMS]) {
    const int G = BH / BHkv, nq = (N + 63) / 64, ntk = (N + 127) / 128;
    const bool edges = window > 0 && window < N;
    const int seen = window > 0 ? (int)std::min<int64_t>(nq, ((int64_t)window + 62) / 64 + 1) : nq;      // 64-key tiles of 64 queries
    const fab::Parts& p = plan.parts;
    auto step_scale = [&](int64_t workgroups) {
        return (1.0 + m.crowd * std::min(1.0, std::max(0.0, (workgroups - 200) / 400.0))) * (edges ? m.edges : 1.0);
    };
    auto dq = [&](Xcd& x, int64_t behind, double scale) {                 // dQ's workgroups behind so many others
        const AttnOrder order{BH, G, G, nq, causal && window <= 0};
        for (int id = (int)(-behind & 7); id < BH * nq; id += 8) {
            int bh, rank, kvbh;
            order.decode(id, bh, rank, kvbh);
            x.run(m.dq_wg + m.dq_tile * scale * (causal ? std::min(nq - rank, seen) : nq));
        }
    };
    us[TWO] = m.two + m.two_dq * attn_us(BH, N, D, causal, window, true) + m.two_dkv * plan.us;
    const double sum = p.chunk ? partial_us(p, BHkv, N, D) : 0.0;
    us[ONE] = us[DS] = us[HALF] = 1e300;
    int64_t items = 0;
    for (int kt = 0; kt < ntk; ++kt) items += p.parts(kt);
    const int64_t one = items * BHkv + (int64_t)BH * nq, half = (int64_t)(BHkv + BH) * nq;
    // Hardly ever the fastest beyond (2 of 1650 shapes); never with whole key tiles and no causal rule at D = 64, where 64-key ones share CUs
    // or two launches do better (0 of 460; B2 H4 N2129 81 us, 69 in two launches)
    if (one <= 1024 && (D == 128 || causal || p.chunk)) {
        Xcd x{8};
        const double scale = step_scale(one), step = m.part_step * scale;
        first_xcd_dkv(p, ntk, BHkv, [&](int steps) { x.run(m.part_wg + step * steps); });
        dq(x, items * BHkv, scale);
        us[ONE] = m.one + x.last + (p.chunk ? m.sum + m.traffic * sum : 0.0);
    }
    const size_t lds = half_lds(D, half_steps(G, N, causal, window), false);
    if (half <= 1600 && lds <= 160 * 1024) {
        const bool shared = D == 64 && lds <= 80 * 1024 && !kept_apart(G, N, causal, window, half);      // CUs, by two workgroups
        Xcd x{shared ? 16 : 8};
        const double beside = shared ? 1.0 + m.beside * std::min(1.0, std::max(0.0, (half - 256) / 256.0)) : 1.0;
        const double scale = step_scale(half) * beside, step = m.half_step * (edges ? scale / m.edges : scale);       // its mask is always on
        const int stride = BHkv % 8 ? 8 : 1, heads = BHkv / (8 / stride);
        for (int at = 0; at < heads * nq; at += stride) {
            const int kt = at / heads;
            x.run(m.half_wg * beside + step * G * (std::min(nq, (window > 0 ? kt : 0) + seen) - (causal ? kt : 0)));
        }
        dq(x, (int64_t)BHkv * nq, scale);
        us[HALF] = m.half + x.last;
    }
    if (D == 128 && ntk > 1 && ds_bytes(BH, N, causal, window) <= kMostDs) {
        // product: stages of 32 keys, two workgroups a CU
        const int longest = 2 * (window > 0 ? (int)std::min<int64_t>(nq, ((int64_t)window + 126) / 64 + 1) : nq);
        double mean = 0;
        for (int qt = 0; qt < ntk; ++qt) mean += causal ? std::min(longest, 4 * (qt + 1)) : longest;
        mean *= BH / 512.0;
        const double scale = edges ? m.edges : 1.0;
        us[DS] = m.ds + m.ds_bytes * (double)BH * N * D * 4 / 1.0e6 + scale * (m.ds_dkv * plan.us + std::max(m.ds_tile * longest, m.ds_mean * mean)) +
                 (p.chunk ? m.ds_sum : 0.0);
    }
}
// some microseconds of host time (tens for hundreds of workgroups): each thread keeps its last plans
struct Launches {
    fab::Parts parts;
    bool wide;                                       // TWO: key tiles of 256 instead
    double us[FORMS];
};
Launches launches(int BH, int BHkv, int N, int D, bool causal, int window, bool cut_tiles) {
    struct Entry { int BH, BHkv, N, D, causal, window, cut; Launches how; };
    static thread_local Entry kept[32];
    const int rule = causal * 2 + cut_tiles;
    const uint32_t h = ((uint32_t)BHkv * 0x9e3779b1u ^ (uint32_t)N * 0x85ebca6bu ^ ((uint32_t)BH * 131u + (uint32_t)D) * 0xc2b2ae35u ^ (uint32_t)(window * 4 + rule) * 0x27d4eb2fu) * 0x9e3779b1u;
    Entry& e = kept[h >> 27];
    if (e.BH != BH || e.BHkv != BHkv || e.N != N || e.D != D || e.causal != causal || e.window != window || e.cut != cut_tiles) {
        const DkvPlan plan = make_dkv_plan(BHkv, BH / BHkv, N, D, causal, window, cut_tiles);
        const double saved = wide_saves(BHkv, BH / BHkv, N, D, causal, window, plan);
        e = {BH, BHkv, N, D, causal, window, cut_tiles, {plan.parts, saved > 0, {}}};
        launch_us(D == 128 ? kModel128 : kModel64, BH, BHkv, N, D, causal, window, plan, e.how.us);
        e.how.us[TWO] -= std::max(0.0, saved);
    }
    return e.how;
}
// What a call does with the scratch it has, and the pieces of that scratch, in this order.  Three forms, each for callers without
// the memory of the next: the pairs alone (whole key tiles), parts too, dS too.  B1 Hq32 Hkv8 N2000: 254 us with 0.5 MiB, 148
// with 32, 136 with 168.
enum class Scratch { Pairs, Parts, Ds };
struct BwdPlan {
    fab::Parts parts;
    int items;
    int64_t dq_blocks, dkv_blocks;                   // dq_blocks: of the 64-row form, beside dK/dV's in one launch
    bool both, ds;
    int half;                                        // half_steps
    size_t stat_bytes, partial_bytes, ds_bytes;
    size_t bytes() const { return stat_bytes + partial_bytes + ds_bytes; }
};
BwdPlan bwd_plan(int B, int Hq, int Hkv, int N, int D, bool causal, int window, Scratch form) {
    BwdPlan p;
    const int BH = B * Hq, BHkv = B * Hkv;
    Launches how = launches(BH, BHkv, N, D, causal, window, form != Scratch::Pairs);
    if (form != Scratch::Ds) how.us[DS] = 1e300;
    const int pick = (int)(std::min_element(how.us, how.us + FORMS) - how.us);
    p.parts = how.parts;
    if (pick == HALF) p.parts.chunk = 0;
    if (pick == TWO && how.wide) {
        p.parts.chunk = 0;
        p.parts.keys = 256;
    }
    p.half = pick == HALF ? half_steps(Hq / Hkv, N, causal, window) : 0;
    p.both = pick == HALF || pick == ONE;
    p.ds = pick == DS;
    p.items = dkv_items(p.parts, N);
    p.dq_blocks = (int64_t)BH * ((N + 63) / 64);
    p.dkv_blocks = (int64_t)BHkv * (p.half ? (N + 63) / 64 : p.items);
    p.stat_bytes = flash_attn_bwd_workspace_bytes(B, Hq, N);
    p.partial_bytes = dkv_partial_bytes(p.parts, B * Hkv, N, D);
    p.ds_bytes = p.ds ? ds_bytes(B * Hq, N, causal, window) : 0;
    return p;
}
}  // namespace

size_t flash_attn_bwd_full_workspace_bytes(int B, int Hq, int Hkv, int N, int D, int causal, int window) {
    return bwd_plan(B, Hq, Hkv, N, D, causal != 0, window, Scratch::Ds).bytes();
}
size_t flash_attn_bwd_parts_workspace_bytes(int B, int Hq, int Hkv, int N, int D, int causal, int window) {
    return bwd_plan(B, Hq, Hkv, N, D, causal != 0, window, Scratch::Parts).bytes();
}

int launch_flash_attn_bwd(const void* q, const void* k, const void* v, const void* o, const void* d_o,
                          const float* lse, void* dq, void* dk, void* dv, int B, int Hq, int Hkv, int N, int D,
                          int causal, int window, const int* kv_lens, const uint8_t* key_mask, float scale,
                          void* workspace, size_t workspace_bytes,
                          hipStream_t stream) {
    using namespace fab;
    const int BH = B * Hq, BHkv = B * Hkv, G = Hq / Hkv;
    const int ntk = (N + 127) / 128, npad = ntk * 128;
    const bool limits = window > 0 || kv_lens != nullptr;     // never together with a key mask
    const AttnShape shape = attn_shape(BH, N, D, causal != 0, window, true);
    const int ntq = (N + shape.rows - 1) / shape.rows;
    const int pair = shape.pair, single = shape.single;
    dim3 grid_q((unsigned)(BH * (pair ? (ntq + 1) / 2 : ntq))), block(THREADS);
    BwdPlan how = bwd_plan(B, Hq, Hkv, N, D, causal != 0, window, Scratch::Ds);
    for (Scratch form : {Scratch::Parts, Scratch::Pairs})
        if (workspace_bytes < how.bytes()) how = bwd_plan(B, Hq, Hkv, N, D, causal != 0, window, form);
    const Parts plan = how.parts;
    const int items = how.items;
    const dim3 grid_k((unsigned)how.dkv_blocks);
    float* partial = reinterpret_cast<float*>(static_cast<unsigned char*>(workspace) + how.stat_bytes);
    unsigned char* ds = static_cast<unsigned char*>(workspace) + how.stat_bytes + how.partial_bytes;
    const float scale_log2 = scale * LOG2E;
    auto Qp = static_cast<const uint16_t*>(q);
    auto Kp = static_cast<const uint16_t*>(k);
    auto Vp = static_cast<const uint16_t*>(v);
    auto Op = static_cast<const uint16_t*>(o);
    auto dOp = static_cast<const uint16_t*>(d_o);
    auto st = static_cast<float2*>(workspace);
#define TYR_FAB_DQ(DD, CC, EE, SS)                                                                    \
    do {                                                                                              \
        static const hipError_t a1 = hipFuncSetAttribute(                                             \
            reinterpret_cast<const void*>(&flash_attn_bwd_dq_kernel<DD, CC, EE, SS>),                 \
            hipFuncAttributeMaxDynamicSharedMemorySize, CfgQ<DD>::LDS);                               \
        if (a1 != hipSuccess) return -1;                                                              \
        launch_kernel((flash_attn_bwd_dq_kernel<DD, CC, EE, SS>), grid_q, block, CfgQ<DD>::LDS, stream, \
                           Qp, Kp, Vp, Op, dOp, lse, static_cast<uint16_t*>(dq), st, BH, N, ntq, npad, \
                           scale, scale_log2, Hq, G, window, kv_lens, key_mask, pair, single, plan.keys == 256 ? 3 : 0); \
    } while (0)
#define TYR_FAB_DKV(DD, CC, EE, UU, PP)                                                               \
    do {                                                                                              \
        static const hipError_t a2 = hipFuncSetAttribute(                                             \
            reinterpret_cast<const void*>(&flash_attn_bwd_dkv_kernel<DD, CC, EE, UU, PP>),            \
            hipFuncAttributeMaxDynamicSharedMemorySize, CfgK<DD>::LDS);                               \
        if (a2 != hipSuccess) return -1;                                                              \
        launch_kernel((flash_attn_bwd_dkv_kernel<DD, CC, EE, UU, PP>), grid_k, block, CfgK<DD>::LDS, \
                           stream, Qp, Kp, Vp, dOp, st, static_cast<uint16_t*>(dk),                   \
                           static_cast<uint16_t*>(dv), BHkv, N, ntk, npad, scale, scale_log2, Hq,     \
                           window, kv_lens, key_mask, plan, items, partial, ds);                      \
    } while (0)
#define TYR_FAB_DKV_WIDE(DD, CC, EE)                                                                  \
    do {                                                                                              \
        static const hipError_t a5 = hipFuncSetAttribute(                                             \
            reinterpret_cast<const void*>(&flash_attn_bwd_dkv_wide_kernel<DD, CC, EE>),               \
            hipFuncAttributeMaxDynamicSharedMemorySize, CfgK<DD>::LDS);                               \
        if (a5 != hipSuccess) return -1;                                                              \
        launch_kernel((flash_attn_bwd_dkv_wide_kernel<DD, CC, EE>), grid_k, block, CfgK<DD>::LDS,     \
                           stream, Qp, Kp, Vp, dOp, st, static_cast<uint16_t*>(dk),                   \
                           static_cast<uint16_t*>(dv), BHkv, N, npad, scale, scale_log2, Hq,          \
                           window, kv_lens, key_mask, plan, items);                                   \
    } while (0)
#define TYR_FAB_DKV_MASK(DD, CC, EE, UU, PP)  /* lengths alone are a mask of keys here; a window is causal */ \
    do {                                                                                              \
        if constexpr (EE == AttnMask::Limits) {                                                       \
            if (CC && window > 0) TYR_FAB_DKV(DD, true, EE, UU, PP);                                  \
            else TYR_FAB_DKV(DD, CC, AttnMask::Keys, UU, PP);                                         \
        } else {                                                                                      \
            TYR_FAB_DKV(DD, CC, EE, UU, PP);                                                          \
        }                                                                                             \
    } while (0)
#define TYR_FAB_DQ_PRODUCT(DD, CC, EE)                                                                \
    do {                                                                                              \
        static const hipError_t a4 = hipFuncSetAttribute(                                             \
            reinterpret_cast<const void*>(&flash_attn_bwd_dq_product_kernel<DD, CC, EE>),             \
            hipFuncAttributeMaxDynamicSharedMemorySize, CfgP<DD>::LDS);                               \
        if (a4 != hipSuccess) return -1;                                                              \
        const int ndq = BH * ntk, nsum = plan.chunk ? BHkv * ntk * (DD / 8) : 0;                      \
        launch_kernel((flash_attn_bwd_dq_product_kernel<DD, CC, EE>), dim3((unsigned)(ndq + nsum)), block, CfgP<DD>::LDS, stream, \
                           Kp, ds, static_cast<uint16_t*>(dq), BH, N, ntk, scale, Hq, window, kv_lens, key_mask, \
                           causal && window <= 0, ndq, partial, static_cast<uint16_t*>(dk),           \
                           static_cast<uint16_t*>(dv), items, plan);                                  \
    } while (0)
#define TYR_FAB_SUM(DD)                                                                               \
    launch_kernel(flash_attn_bwd_sum_kernel<DD>, dim3((unsigned)(BHkv * ntk * (DD / 8))), dim3(256), 0, stream, \
                       partial, static_cast<uint16_t*>(dk), static_cast<uint16_t*>(dv), N, ntk, items, scale, plan)
#define TYR_FAB_BOTH(DD, CC, EE, UU, HH)                                                               \
    do {                                                                                              \
        static const hipError_t a3 = hipFuncSetAttribute(                                             \
            reinterpret_cast<const void*>(&flash_attn_bwd_both_kernel<DD, CC, EE, UU, HH>),               \
            hipFuncAttributeMaxDynamicSharedMemorySize, HH ? 160 * 1024 : CfgK<DD>::LDS);                               \
        if (a3 != hipSuccess) return -1;                                                              \
        launch_kernel((flash_attn_bwd_both_kernel<DD, CC, EE, UU, HH>), dim3((unsigned)(how.dkv_blocks + how.dq_blocks)), block, HH ? half_lds(DD, how.half, kept_apart(G, N, causal, window, how.dkv_blocks + how.dq_blocks)) : CfgK<DD>::LDS, \
                           stream, Qp, Kp, Vp, Op, dOp, lse, static_cast<uint16_t*>(dq), st,          \
                           static_cast<uint16_t*>(dk), static_cast<uint16_t*>(dv), BH, N, (N + 63) / 64, ntk, \
                           npad, scale, scale_log2, Hq, window, kv_lens, key_mask, causal && window <= 0, plan, items, partial, (int)how.dkv_blocks); \
    } while (0)
#define TYR_FAB_LAUNCH(DD, CC, EE)                                                                    \
    do {                                                                                              \
        if (how.both) {                                                                               \
            if (how.half) { TYR_FAB_BOTH(DD, CC, EE, false, true); break; }                           \
            if (!plan.chunk) {                                                                        \
                if constexpr (DD == 128 || CC) TYR_FAB_BOTH(DD, CC, EE, false, false);                \
                break;                                                                                \
            }                                                                                         \
            TYR_FAB_BOTH(DD, CC, EE, true, false);                                                    \
            TYR_FAB_SUM(DD);                                                                          \
            break;                                                                                    \
        }                                                                                             \
        if constexpr (DD == 128) {                                                                               \
            if (how.ds) {                                                                             \
                launch_kernel(flash_attn_bwd_stats_kernel<DD>, dim3((unsigned)(BH * (npad / (2048 / DD)))), dim3(256), 0, \
                                   stream, Op, dOp, lse, st, N, npad, EE != AttnMask::None);          \
                if (plan.chunk) TYR_FAB_DKV_MASK(DD, CC, EE, true, true);                             \
                else TYR_FAB_DKV_MASK(DD, CC, EE, false, true);                                       \
                TYR_FAB_DQ_PRODUCT(DD, CC, EE);                                                       \
                break;                                                                                \
            }                                                                                         \
        }                                                                                             \
        if (shape.rows == 64) TYR_FAB_DQ(DD, CC, EE, true); else TYR_FAB_DQ(DD, CC, EE, false);       \
        if (plan.keys == 256) {                                                                       \
            if constexpr (EE == AttnMask::Limits) {                                                   \
                if (CC && window > 0) TYR_FAB_DKV_WIDE(DD, true, EE);                                 \
                else TYR_FAB_DKV_WIDE(DD, CC, AttnMask::Keys);                                        \
            } else {                                                                                  \
                TYR_FAB_DKV_WIDE(DD, CC, EE);                                                         \
            }                                                                                         \
            break;                                                                                    \
        }                                                                                             \
        if (plan.chunk) {                                                                             \
            TYR_FAB_DKV_MASK(DD, CC, EE, true, false);                                                \
            TYR_FAB_SUM(DD);                                                                          \
        } else {                                                                                      \
            TYR_FAB_DKV_MASK(DD, CC, EE, false, false);                                               \
        }                                                                                             \
    } while (0)
#define TYR_FAB_PICK(DD, MM)                                                                          \
    do { if (causal) TYR_FAB_LAUNCH(DD, true, MM); else TYR_FAB_LAUNCH(DD, false, MM); } while (0)
#define TYR_FAB_MASK(DD)                                                                              \
    do {                                                                                              \
        if (key_mask != nullptr) TYR_FAB_PICK(DD, AttnMask::Keys);                                    \
        else if (limits) TYR_FAB_PICK(DD, AttnMask::Limits);                                          \
        else TYR_FAB_PICK(DD, AttnMask::None);                                                        \
    } while (0)
    if (D == 128) TYR_FAB_MASK(128); else TYR_FAB_MASK(64);
#undef TYR_FAB_MASK
#undef TYR_FAB_PICK
#undef TYR_FAB_LAUNCH
#undef TYR_FAB_BOTH
#undef TYR_FAB_SUM
#undef TYR_FAB_DQ_PRODUCT
#undef TYR_FAB_DKV_MASK
#undef TYR_FAB_DKV
#undef TYR_FAB_DKV_WIDE
#undef TYR_FAB_DQ
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace tyr
