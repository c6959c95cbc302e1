// The two launches that end a training step of the surrogate, after the backward pass has left
// every layer's dZ: all gradients (grads_body), then their final sums and Adam (update_body).
//
// grads_body gives each block one of three jobs:
//   * a 128 x 128 tile of one split of one layer's weight gradient (gemm_tn_body);
//   * four rows of a hidden layer's bias gradient: wave t sums rows t, t + 256, ... of dZ for all
//     256 columns, four neighbouring columns a lane, so a wave reads whole 512-byte rows (one
//     block per column, two bytes a lane from 512-byte strides, took 100 us a layer at 65536
//     rows: every lane's load fetched a cache line of its own);
//   * two rows of the output layer's gradient, split over the batch the same way.
// The sums' jobs come first in the grid: they are serial chains of rows / 256 additions, a few
// waves wide, and run beside the matrix tiles.  What bounds the launch: reading every layer's
// input and dZ once for the tiles and once for the sums.  65536 rows: 107 us for all of it, where
// a launch per layer and sum took 138 us x 4 (generic tiles), 100 us x 4 and 167 us.
//
// update_body finishes the sums and applies Adam to each parameter as its gradient becomes
// known: a weight adds its split partials in ascending order; a bias and an output-layer weight
// add their 256 row sums as a binary tree (t, t + 128), (t, t + 64), ...  One launch for all
// ten parameter arrays: each is too small to fill the device (a bias is one block).  18 us at 64
// splits (the partials' 65 MB), where four reductions and ten Adam launches took 113.
#pragma once
#include "gemm_tn.hpp"
#include "mlp_fused.hpp"

namespace lm {

#define LM_SUM_ROWS 256                      // row sums kept per column: rows t, t + 256, ...
#define LM_COL_BLOCKS (LM_SUM_ROWS / 4)      // blocks of one layer's column sums (one wave a t)
#define LM_OUT_BLOCKS (LM_SUM_ROWS / 2)      // blocks of the output layer's sums (two waves a t)

struct GradParams {
    GemmParams dw[4];      // dW of the hidden layers: A = the layer's input, B = its dZ, out_f32 = partials
    int splits;
    int rows;              // mini-batch rows
    const u16* act_top;    // [rows][256] the last hidden layer's activations
    const float* dout;     // [rows][LS_OUT]
    float* col_part;       // [4][256 t][256] row sums of dZ
    float* out_part;       // [256 t][257][LS_OUT] row sums of act x dOut, and of dOut (row 256)
};

// Sums of rows t, t + 256, ... of dZ [rows][256]: four columns a lane.
__device__ __forceinline__ void column_sums_body(const u16* dz, int rows, int t, float* part) {
    const int lane = threadIdx.x & 63;
    const u16* p = dz + 4 * lane;
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    auto add = [&](uint2 x) {
        s[0] += __uint_as_float(x.x << 16);
        s[1] += __uint_as_float(x.x & 0xffff0000u);
        s[2] += __uint_as_float(x.y << 16);
        s[3] += __uint_as_float(x.y & 0xffff0000u);
    };
    int i = t;
    for (; i + 15 * LM_SUM_ROWS < rows; i += 16 * LM_SUM_ROWS) {  // 16 rows in flight
        uint2 x[16];
#pragma unroll
        for (int u = 0; u < 16; ++u)
            x[u] = *reinterpret_cast<const uint2*>(p + (size_t)(i + u * LM_SUM_ROWS) * LS_HIDDEN);
#pragma unroll
        for (int u = 0; u < 16; ++u) add(x[u]);
    }
    for (; i < rows; i += LM_SUM_ROWS) add(*reinterpret_cast<const uint2*>(p + (size_t)i * LS_HIDDEN));
    *reinterpret_cast<float4*>(part + (size_t)t * LS_HIDDEN + 4 * lane) = make_float4(s[0], s[1], s[2], s[3]);
}

// Sums over rows t, t + 256, ... of act[i][k] dOut[i][o] for k = 128 half + 2 lane and the next
// one, and (half 0) of dOut[i][o] for the bias.
__device__ __forceinline__ void out_layer_sums_body(const u16* act, const float* dout, int rows, int t, int half,
                                                    float* part) {
    const int lane = threadIdx.x & 63;
    const int k = 128 * half + 2 * lane;
    float s0[LS_OUT], s1[LS_OUT], sb[LS_OUT];
#pragma unroll
    for (int o = 0; o < LS_OUT; ++o) s0[o] = s1[o] = sb[o] = 0.0f;
    auto add = [&](unsigned a, const float* d) {
        const float a0 = __uint_as_float(a << 16), a1 = __uint_as_float(a & 0xffff0000u);
#pragma unroll
        for (int o = 0; o < LS_OUT; ++o) {
            s0[o] = __builtin_fmaf(a0, d[o], s0[o]);
            s1[o] = __builtin_fmaf(a1, d[o], s1[o]);
            sb[o] += d[o];
        }
    };
    int i = t;
    for (; i + 7 * LM_SUM_ROWS < rows; i += 8 * LM_SUM_ROWS) {  // 8 rows in flight
        unsigned a[8];
        float d[8][LS_OUT];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const size_t r = (size_t)(i + u * LM_SUM_ROWS);
            a[u] = *reinterpret_cast<const unsigned*>(act + r * LS_HIDDEN + k);
#pragma unroll
            for (int o = 0; o < LS_OUT; ++o) d[u][o] = dout[r * LS_OUT + o];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) add(a[u], d[u]);
    }
    for (; i < rows; i += LM_SUM_ROWS) {
        float d[LS_OUT];
#pragma unroll
        for (int o = 0; o < LS_OUT; ++o) d[o] = dout[(size_t)i * LS_OUT + o];
        add(*reinterpret_cast<const unsigned*>(act + (size_t)i * LS_HIDDEN + k), d);
    }
    float* out = part + (size_t)t * (LS_HIDDEN + 1) * LS_OUT;
#pragma unroll
    for (int o = 0; o < LS_OUT; ++o) {
        out[k * LS_OUT + o] = s0[o];
        out[(k + 1) * LS_OUT + o] = s1[o];
        if (half == 0 && lane == 0) out[LS_HIDDEN * LS_OUT + o] = sb[o];
    }
}

__host__ __device__ inline int grads_sum_blocks() { return 4 * LM_COL_BLOCKS + LM_OUT_BLOCKS; }
__host__ __device__ inline int grads_tiles(const GradParams& P) {
    return P.splits * (gemm_tn_tiles(P.dw[0]) + gemm_tn_tiles(P.dw[1]) + gemm_tn_tiles(P.dw[2]) + gemm_tn_tiles(P.dw[3]));
}

__device__ __forceinline__ void grads_body(const GradParams& P) {
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    int b = blockIdx.x;
    if (b < 4 * LM_COL_BLOCKS) {
        const int l = b / LM_COL_BLOCKS, t = (b % LM_COL_BLOCKS) * 4 + wave;
        column_sums_body(P.dw[l].B, P.rows, t, P.col_part + (size_t)l * LM_SUM_ROWS * LS_HIDDEN);
        return;
    }
    b -= 4 * LM_COL_BLOCKS;
    if (b < LM_OUT_BLOCKS) {
        out_layer_sums_body(P.act_top, P.dout, P.rows, 2 * b + (wave >> 1), wave & 1, P.out_part);
        return;
    }
    int work = gemm_tn_work(b - LM_OUT_BLOCKS, grads_tiles(P));  // both sums' block counts are multiples of 8
    int l = 0;
    for (; l < 3; ++l) {
        const int n = P.splits * gemm_tn_tiles(P.dw[l]);
        if (work < n) break;
        work -= n;
    }
    gemm_tn_body(P.dw[l], work);
}

// ---- Adam ----------------------------------------------------------------------------------
struct AdamStep {
    float lr, b1, b2, eps, bc1, bc2;
};

// One parameter's update, with its contractions written out (so that every kernel rounds it the
// same way); returns the new value.
__device__ __forceinline__ float adam_update(const AdamStep& A, float g, float* w, float* m, float* v) {
#pragma clang fp contract(off)
    const float mm = __builtin_fmaf(1.0f - A.b1, g, A.b1 * *m);
    const float vv = __builtin_fmaf(g, (1.0f - A.b2) * g, A.b2 * *v);
    *m = mm;
    *v = vv;
    const float nw = *w - A.lr * (mm / A.bc1) / (sqrtf(vv / A.bc2) + A.eps);
    *w = nw;
    return nw;
}

struct LayerUpdate {
    float *w, *m, *v;     // [K][256]
    float *b, *mb, *vb;   // [256]
    u16* wpack;           // the BF16 fragments of the forward product (mlp_pack_body's order)
    u16* bpack;           // and of the backward product, W^T; null for the first layer
    const float* part;    // [splits][K][256]
    int K;
};
struct UpdateParams {
    LayerUpdate hidden[4];
    float *w, *m, *v;     // output layer [256][LS_OUT]
    float *b, *mb, *vb;   // [LS_OUT]
    const float* col_part;
    const float* out_part;
    int splits;
    AdamStep adam;
};

__host__ __device__ inline int update_blocks(const UpdateParams& P) {
    return P.hidden[0].K + P.hidden[1].K + P.hidden[2].K + P.hidden[3].K + 4 * LS_HIDDEN / 4 + LS_HIDDEN + 1;
}

// The tree over the 256 row sums of C columns, one thread per row sum; the totals in red[.][0].
template <int C>
__device__ __forceinline__ void sum_tree(float (&red)[C][LM_SUM_ROWS]) {
    const int t = threadIdx.x;
    __syncthreads();
    for (int st = LM_SUM_ROWS / 2; st > 0; st >>= 1) {
        if (t < st)
            for (int c = 0; c < C; ++c) red[c][t] += red[c][t + st];
        __syncthreads();
    }
}

// Blocks of LM_SUM_ROWS threads: one per hidden weight row k, then one per four hidden biases,
// then one per output-layer row (the last: its bias).
__device__ __forceinline__ void update_body(const UpdateParams& P) {
    __shared__ float red[LS_OUT][LM_SUM_ROWS];
    const int t = threadIdx.x;
    int b = blockIdx.x;
    for (int l = 0; l < 4; ++l) {
        const LayerUpdate& L = P.hidden[l];
        if (b < L.K) {
            const size_t j = (size_t)b * LS_HIDDEN + t, stride = (size_t)L.K * LS_HIDDEN;
            const float* p = L.part + j;
            float g = 0.0f;
            int s = 0;
            for (; s + 16 <= P.splits; s += 16) {
                float x[16];
#pragma unroll
                for (int u = 0; u < 16; ++u) x[u] = p[(size_t)(s + u) * stride];
#pragma unroll
                for (int u = 0; u < 16; ++u) g += x[u];
            }
            for (; s < P.splits; ++s) g += p[(size_t)s * stride];
            const float nw = adam_update(P.adam, g, L.w + j, L.m + j, L.v + j);
            const u16 nb = f2bf(nw);
            L.wpack[pack_index(b, t)] = nb;
            if (L.bpack) L.bpack[pack_index(t, b)] = nb;
            return;
        }
        b -= L.K;
    }
    if (b < LS_HIDDEN) {  // four biases of one layer
        const int l = b >> 6, c0 = 4 * (b & 63);
        const float4 x = *reinterpret_cast<const float4*>(P.col_part + ((size_t)l * LM_SUM_ROWS + t) * LS_HIDDEN + c0);
        float(&r4)[4][LM_SUM_ROWS] = reinterpret_cast<float(&)[4][LM_SUM_ROWS]>(red);
        r4[0][t] = x.x;
        r4[1][t] = x.y;
        r4[2][t] = x.z;
        r4[3][t] = x.w;
        sum_tree(r4);
        const LayerUpdate& L = P.hidden[l];
        if (t < 4) adam_update(P.adam, r4[t][0], L.b + c0 + t, L.mb + c0 + t, L.vb + c0 + t);
        return;
    }
    const int k = b - LS_HIDDEN;  // an output-layer row; LS_HIDDEN: its bias
    const float* p = P.out_part + ((size_t)t * (LS_HIDDEN + 1) + k) * LS_OUT;
    for (int o = 0; o < LS_OUT; ++o) red[o][t] = p[o];
    sum_tree(red);
    if (t < LS_OUT) {
        const int j = k * LS_OUT + t;
        if (k < LS_HIDDEN)
            adam_update(P.adam, red[t][0], P.w + j, P.m + j, P.v + j);
        else
            adam_update(P.adam, red[t][0], P.b + t, P.mb + t, P.vb + t);
    }
}

}  // namespace lm
