// Fast path of the surrogate GEMM for a weight gradient, dW = X^T dZ over a mini-batch: both
// operands are stored with the contraction (the batch rows) as the slow index, A [K][M] and
// B [K][N], and the batch is split into chunks whose FP32 partials are summed afterwards.
//   * block tile 128 x 128, 4 waves, each wave 64 x 64 = 2 x 2 v_mfma_f32_32x32x16_bf16 tiles;
//   * batch rows in steps of 32: a lane loads two neighbouring columns of 8 rows of A and of B
//     (4 B each; a wave's load is 256 contiguous bytes of one row), transposes them in registers
//     (v_perm_b32 pairs rows of one column) and writes 8 consecutive rows of a column to LDS as
//     one 16-byte store, the [column][row] order the MFMA operands are read in;
//   * two LDS buffers and two register sets: the loads of a step are issued two steps ahead;
//   * the tiles of one split follow one another on one XCD, whose L2 then holds the chunk's rows
//     for all of them.
// What bounds it: the latency of the row loads (a chunk is 1024 rows, 32 steps a block) and LDS
// reads, 16 KB per 4 MFMAs of a CU's four waves, 128 B a cycle.  At 65536 rows and 256 x 256
// outputs (64 chunks, 256 blocks) it takes 24.6 us; gemm_body, with its 2-byte loads and stores, 138 us.
// The k order is gemm_body's (ascending steps of 16 into one accumulator), so the partials are
// the same bits.
// Requires K and the chunk to be multiples of 32, N % 128 == 0, and even M, lda and ldb.
#pragma once
#include "mlp.hpp"

namespace lm {

#define LM_TN_BM 128
#define LM_TN_BN 128
#define LM_TN_BK 32
#define LM_TN_LD (LM_TN_BK + 8)
#define LM_TN_XCDS 8

__host__ __device__ inline bool gemm_tn_applies(const GemmParams& P) {
    return P.a_trans && !P.b_trans && P.epi == LM_EPI_PARTIAL && (P.K % LM_TN_BK) == 0 &&
           (P.k_per_split % LM_TN_BK) == 0 && (P.N % LM_TN_BN) == 0 && (P.M % 2) == 0 && (P.lda % 2) == 0 &&
           (P.ldb % 2) == 0;
}
__host__ __device__ inline int gemm_tn_tiles(const GemmParams& P) {
    return ((P.M + LM_TN_BM - 1) / LM_TN_BM) * (P.N / LM_TN_BN);
}

// block b of tiles x splits: consecutive b go to the XCDs in turn, and each XCD takes a
// contiguous run of (split, tile) pairs
__device__ __forceinline__ int gemm_tn_work(int b, int n) {
    const int q = n / LM_TN_XCDS, r = n % LM_TN_XCDS;
    const int x = b % LM_TN_XCDS, i = b / LM_TN_XCDS;
    return x * q + min(x, r) + i;
}

__device__ __forceinline__ void gemm_tn_body(const GemmParams& P, int work) {
    typedef unsigned int u32x4t __attribute__((ext_vector_type(4)));
    __shared__ __attribute__((aligned(16))) u16 sA[2][LM_TN_BM][LM_TN_LD];
    __shared__ __attribute__((aligned(16))) u16 sB[2][LM_TN_BN][LM_TN_LD];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int tiles_n = P.N / LM_TN_BN, tiles = gemm_tn_tiles(P);
    const int split = work / tiles, tile = work % tiles;
    const int m0 = (tile / tiles_n) * LM_TN_BM, n0 = (tile % tiles_n) * LM_TN_BN;
    const int kbeg = split * P.k_per_split;
    const int kend = min(P.K, kbeg + P.k_per_split);
    const int nk = (kend - kbeg) / LM_TN_BK;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    // this lane's columns (2 lane, 2 lane + 1) of rows 8 wave .. +7 of each step; M is even, so a
    // column pair is inside or outside as a whole
    const bool a_in = m0 + 2 * lane < P.M;
    const unsigned la = a_in ? (unsigned)(m0 + 2 * lane) : 0u, lb = (unsigned)(n0 + 2 * lane);
    const u16* pa = P.A + (size_t)(kbeg + 8 * wave) * P.lda;  // wave-uniform: the loads take a scalar base
    const u16* pb = P.B + (size_t)(kbeg + 8 * wave) * P.ldb;
    struct Rows {
        unsigned a[8], b[8];
    };
    auto load = [&](int step, Rows& x) {
        const u16* a = pa + (size_t)step * LM_TN_BK * P.lda;
        const u16* b = pb + (size_t)step * LM_TN_BK * P.ldb;
#pragma unroll
        for (int r = 0; r < 8; ++r) x.a[r] = *reinterpret_cast<const unsigned*>(a + (size_t)r * P.lda + la);
#pragma unroll
        for (int r = 0; r < 8; ++r) x.b[r] = *reinterpret_cast<const unsigned*>(b + (size_t)r * P.ldb + lb);
        // keep the loads here: the scheduler would otherwise sink them next to their use
        __builtin_amdgcn_sched_barrier(0);
    };
    auto put = [&](u16 (*dst)[LM_TN_LD], const unsigned (&x)[8]) {
        u32x4t lo, hi;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            lo[q] = __builtin_amdgcn_perm(x[2 * q + 1], x[2 * q], 0x05040100u);
            hi[q] = __builtin_amdgcn_perm(x[2 * q + 1], x[2 * q], 0x07060302u);
        }
        *reinterpret_cast<u32x4t*>(&dst[2 * lane][8 * wave]) = lo;
        *reinterpret_cast<u32x4t*>(&dst[2 * lane + 1][8 * wave]) = hi;
    };
    auto store = [&](int buf, Rows& x) {
        if (!a_in) {
#pragma unroll
            for (int r = 0; r < 8; ++r) x.a[r] = 0u;
        }
        put(sA[buf], x.a);
        put(sB[buf], x.b);
    };
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    auto compute = [&](int buf) {
#pragma unroll
        for (int ks = 0; ks < LM_TN_BK; ks += 16) {
            const int kq = ks + 8 * (lane >> 5);
            bf16x8 fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                fa[i] = *reinterpret_cast<const bf16x8*>(&sA[buf][wm + 32 * i + (lane & 31)][kq]);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                fb[j] = *reinterpret_cast<const bf16x8*>(&sB[buf][wn + 32 * j + (lane & 31)][kq]);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
    };

    // the steps past the last reload it (never used): with unconditional loads as many are in
    // flight on every path, so the waits before the stores count exactly
    Rows r0, r1;
    load(0, r0);
    load(min(1, nk - 1), r1);
    store(0, r0);
    __syncthreads();
    for (int it = 0; it + 1 < nk; it += 2) {
        load(min(it + 2, nk - 1), r0);
        compute(0);
        store(1, r1);
        __syncthreads();
        load(min(it + 3, nk - 1), r1);
        compute(1);
        store(0, r0);
        __syncthreads();
    }
    if (nk & 1) compute(0);

    float* out = P.out_f32 + (size_t)split * P.M * P.N;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int col = n0 + wn + 32 * j + (lane & 31);
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = m0 + wm + 32 * i + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
                if (row < P.M) out[(size_t)row * P.N + col] = acc[i][j][e];
            }
        }
}

}  // namespace lm
