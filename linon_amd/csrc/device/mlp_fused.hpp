// Fused inference of the surrogate MLP: Fourier features, the four hidden layers and the FP32
// output layer for a tile of 128 rays in one workgroup, activations kept in LDS between layers.
//
//   * 256 threads = 4 waves; wave w computes all 128 rays for columns 64 w .. +63 of each hidden
//     layer as 2 x 4 tiles of v_mfma_f32_32x32x16_bf16 (128 accumulators per lane), so every
//     weight fragment is loaded by one wave of the workgroup.
//   * Layer input: bf16 [128][264] in LDS (264 = 256 + 8 bf16 of padding, so consecutive rows
//     start 16 B apart in the bank space); each lane reads its 8 consecutive k of one ray with
//     one 16-byte LDS read.
//   * Weights: prepacked once per weight update in MFMA fragment order ([k/16][column
//     tile][lane][8 bf16], see mlp_pack_body), so a wave's fragment is one contiguous, coalesced
//     1 KB global load (L2 resident: 496 KB for all four layers), two k steps ahead of the
//     MFMAs that use it, over the layers' borders too.
//   * Epilogue: bias + SiLU, rounded to bf16 into the same LDS tile after a barrier, 4 columns
//     of a ray per 8-byte LDS write; the biases of all layers wait in LDS.  The last hidden layer
//     is followed by the FP32 output layer (256 -> 7) from LDS, on 4x4x1 FP32 MFMAs (mlp_output).
//   * 80,000 bytes of LDS and 232 registers: two workgroups a CU, whose waves share a SIMD, one's
//     epilogue (about 5,000 cycles a layer, the exponential and the reciprocal quarter rate) beside
//     the other's MFMAs (4,100).
// What bounds it: those VALU instructions.  While MFMAs run beside them the epilogue takes 7,600
// cycles, so that two workgroups held in opposite phases by common barriers (one of 512 threads)
// gain 4% at 8,192 tiles and lose 6% at 1,563, where the last round is nearly empty; raised
// priority of either phase loses 5-15%.  1,048,576 rays 0.72 -> 0.65 ms (820 TFLOP/s), 200,000 rays
// 157 -> 144 us, one round of tiles 30.4 -> 25.5 us (before: weights and output weights read as
// they were needed, cleared accumulators, 2-byte feature writes).
//
// The arithmetic is the unfused path's (features_body, gemm_nt_body with the bias-SiLU
// epilogue, out_layer_kernel): the same roundings in the same order (k in ascending steps of 16
// into one accumulator, sequential FMA over k in the output layer), so both give the same bits.
#pragma once
#include "mlp.hpp"
#include "surrogate.hpp"

namespace lm {

#define LM_FUSED_ROWS 128
#define LM_FUSED_LDA (LS_HIDDEN + 8)
#define LM_FUSED_W5 (LS_HIDDEN + 4)
#define LM_FUSED_KSTEPS0 (LS_FEATS_PAD / 16)     // 14 k steps of the first layer
#define LM_FUSED_KSTEPS (LS_HIDDEN / 16)         // 16 k steps of the others
// bf16 elements of the packed weights of one layer
#define LM_PACK_LAYER0 (LS_FEATS_PAD * LS_HIDDEN)
#define LM_PACK_LAYER (LS_HIDDEN * LS_HIDDEN)
#define LM_PACK_TOTAL (LM_PACK_LAYER0 + 3 * LM_PACK_LAYER)

__host__ __device__ inline size_t pack_offset(int layer) {
    return layer == 0 ? 0 : (size_t)LM_PACK_LAYER0 + (size_t)(layer - 1) * LM_PACK_LAYER;
}

// A hidden layer's weights in MFMA fragment order: element e of fragment (ks, ct, lane) is what
// lane `lane` supplies for the k step ks of column tile ct, the value of contraction index
// 16 ks + 8 (lane / 32) + e and column 32 ct + lane % 32.  Where (k, n) stands:
__host__ __device__ inline int pack_index(int k, int n) {
    return (((k >> 4) * 8 + (n >> 5)) * 64 + (n & 31) + 32 * ((k >> 3) & 1)) * 8 + (k & 7);
}

// Packs one hidden layer's FP32 master weights W [K][256] as BF16 fragments, one thread per
// fragment: of the forward product (contraction over k), or, with Transposed, of the backward
// product W^T (contraction over the 256 columns; K = 256).
template <bool Transposed>
__device__ __forceinline__ void mlp_pack_body(const float* W, int K, u16* dst) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (K / 16) * 8 * 64) return;
    const int lane = t & 63, ct = (t >> 6) & 7, ks = t >> 9;
    const int k0 = 16 * ks + 8 * (lane >> 5), n = 32 * ct + (lane & 31);
    for (int e = 0; e < 8; ++e)
        dst[(size_t)t * 8 + e] = f2bf(Transposed ? W[(size_t)n * LS_HIDDEN + k0 + e] : W[(size_t)(k0 + e) * LS_HIDDEN + n]);
}

struct MlpInferParams {
    const float* states;  // [n][6] entry states (p, q)
    int n;
    float radius;
    const float* freqs;   // [LS_FREQS]
    const u16* wpack;     // LM_PACK_TOTAL packed hidden weights
    const float* bias[4]; // hidden-layer biases [256]
    const float* w_out;   // [256][LS_OUT] FP32
    const float* b_out;   // [LS_OUT]
    float* out;           // [n][LS_OUT]
    const int* n_dev;     // optional: n on the device (then n is the launch's capacity)
};

typedef unsigned int u32x4v __attribute__((ext_vector_type(4)));
typedef float f32x4v __attribute__((ext_vector_type(4)));

// This wave's weight fragments of k steps ks and ks + 1.
__device__ __forceinline__ void mlp_load_pair(const u16* wl, int ks, int wave, int lane, u32x4v (&w)[2][2]) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 2; ++j)
            w[h][j] = *reinterpret_cast<const u32x4v*>(wl + ((size_t)((ks + h) * 8 + 2 * wave + j) * 64 + lane) * 8);
}

template <int V>
struct IntType {
    static constexpr int value = V;
};

// The k loop of one hidden layer, acc = the layer's products: this wave's weight fragments (column
// tiles 2 wave and 2 wave + 1 of each k step, 1 KB each) are loaded two k steps ahead of the MFMAs
// that use them, in two register sets that pairs of steps use in turn; the activations' fragments
// one step ahead.  w0 holds the fragments of steps 0 and 1 on entry; the last pair loads those of
// `next`, the following layer, into w0 (an even number of pairs) or w1, so that no layer begins
// with the latency of L2 (Next; a caller without the registers to hold them loads them before each
// layer).  The first step's MFMAs take the constant zero for their C operand.
template <int KSTEPS, bool Next>
__device__ __forceinline__ void mlp_layer_k(const u16* wl, const u16* next, const u16 (*act)[LM_FUSED_LDA], int wave,
                                            int lane, f32x16 (&acc)[2][4], u32x4v (&w0)[2][2], u32x4v (&w1)[2][2]) {
    static_assert(KSTEPS % 2 == 0, "k steps come in pairs");
    constexpr int PAIRS = KSTEPS / 2;
    const u16* arow = &act[lane & 31][8 * (lane >> 5)];
    bf16x8 x[2][4];
    auto read = [&](int ks, bf16x8 (&v)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const bf16x8*>(arow + 32 * i * LM_FUSED_LDA + 16 * ks);
    };
    read(0, x[0]);
#pragma unroll
    for (int p = 0; p < PAIRS; ++p) {
        u32x4v(&w)[2][2] = p & 1 ? w1 : w0;
        if (Next || p + 1 < PAIRS)
            mlp_load_pair(p + 1 < PAIRS ? wl : next, p + 1 < PAIRS ? 2 * (p + 1) : 0, wave, lane, p & 1 ? w0 : w1);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int ks = 2 * p + h;
            if (ks + 1 < KSTEPS) read(ks + 1, x[(ks + 1) & 1]);
            // the loads stay ahead of this step's MFMAs: the scheduler would sink them to their use
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                bf16x8 wv;
                __builtin_memcpy(&wv, &w[h][j], 16);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv, x[ks & 1][i], ks ? acc[j][i] : f32x16{}, 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// Half of the features of a ray's entry state (features_body's arithmetic), eight frequencies, into
// its row o of the LDS tile; zeros without a state.  A sine and its cosine are neighbours: one
// conversion and one 4-byte write.
__device__ __forceinline__ void mlp_features(const float* state, float radius, const float* freqs, int half, u16* o) {
    unsigned* o2 = reinterpret_cast<unsigned*>(o);
    if (state) {
        float x[LS_IN];
        const float inv_r = 1.0f / radius;
        for (int k = 0; k < 3; ++k) x[k] = state[k] * inv_r;
        for (int k = 3; k < 6; ++k) x[k] = state[k];
        if (half == 0)
            for (int k = 0; k < LS_IN; k += 2) o2[k / 2] = f2bf2(x[k], x[k + 1]);
        float w[8];  // read before the loop: a read a frequency is a wait each
#pragma unroll
        for (int f = 0; f < 8; ++f) w[f] = freqs[8 * half + f];
#pragma unroll
        for (int f = 0; f < 8; ++f)
#pragma unroll
            for (int k = 0; k < LS_IN; ++k) {
                float s, c;
                __sincosf(w[f] * x[k], &s, &c);
                o2[LS_IN / 2 + (8 * half + f) * LS_IN + k] = f2bf2(s, c);
            }
        if (half == 1)
            for (int k = LS_FEATS / 2; k < LS_FEATS_PAD / 2; ++k) o2[k] = 0;
    } else {
        for (int k = half; k < LS_FEATS_PAD / 2; k += 2) o2[k] = 0;
    }
}

// Output layer: outputs o0 .. o0 + 3 (o0 0 or 4, the eighth is zero) of a ray a lane, from the ray's
// last activations and the weights w5 [output][k] in LDS.  One v_mfma_f32_4x4x1_16b_f32 a k: lane l
// supplies its ray's activation and the weight of output o0 + l % 4, and its accumulator's four
// registers are its ray's four outputs, one fused multiply-add each, k ascending: the bits of the FMA
// sequence it stands for.  (That needs a broadcast weight per FMA: 256 16-byte LDS reads a wave, or
// scalar loads with a wait for every few, which took 17,000 cycles of a tile's 70,000; here 256 times
// an MFMA's latency of 14.)
__device__ __forceinline__ f32x4v mlp_output(const u16* arow, const float (*w5)[LM_FUSED_W5], int o0, int lane) {
    f32x4v s;
#pragma unroll
    for (int q = 0; q < 4; ++q) s[q] = w5[o0 + q][LS_HIDDEN];
    const float* wrow = w5[o0 + (lane & 3)];
#pragma unroll
    for (int k8 = 0; k8 < LS_HIDDEN; k8 += 8) {
        const uint4 a8 = *reinterpret_cast<const uint4*>(arow + k8);
        const unsigned aw[4] = {a8.x, a8.y, a8.z, a8.w};
        const float4 wa = *reinterpret_cast<const float4*>(wrow + k8), wb = *reinterpret_cast<const float4*>(wrow + k8 + 4);
        const float w[8] = {wa.x, wa.y, wa.z, wa.w, wb.x, wb.y, wb.z, wb.w};
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) {
            const float a = __uint_as_float(kk & 1 ? (aw[kk >> 1] & 0xffff0000u) : (aw[kk >> 1] << 16));
            s = __builtin_amdgcn_mfma_f32_4x4x1f32(w[kk], a, s, 0, 0, 0);
        }
    }
    return s;
}

// w5 [output][k] from the master weights [k][output], the eighth output zero, and behind each row its
// bias; thread k of LS_HIDDEN.
__device__ __forceinline__ void mlp_stage_output(const float* w_out, const float* b_out, float (*w5)[LM_FUSED_W5], int k) {
    float w[LS_OUT];
#pragma unroll
    for (int o = 0; o < LS_OUT; ++o) w[o] = w_out[k * LS_OUT + o];
#pragma unroll
    for (int o = 0; o < LS_OUT; ++o) w5[o][k] = w[o];
    w5[LS_OUT][k] = 0.0f;
    if (k < 8) w5[k][LS_HIDDEN] = k < LS_OUT ? b_out[k] : 0.0f;
}

__device__ __forceinline__ void mlp_infer_body(const MlpInferParams& P) {
    __shared__ __attribute__((aligned(16))) u16 act[LM_FUSED_ROWS][LM_FUSED_LDA];
    __shared__ __attribute__((aligned(16))) float bias[4][LS_HIDDEN];
    __shared__ __attribute__((aligned(16))) float w5[8][LM_FUSED_W5];
    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int row0 = blockIdx.x * LM_FUSED_ROWS;
    const int n = P.n_dev ? *P.n_dev : P.n;
    if (row0 >= n) return;  // whole workgroup, before any barrier
    u32x4v wa[2][2], wb[2][2];
    mlp_load_pair(P.wpack, 0, wave, lane, wb);
#pragma unroll
    for (int l = 0; l < 4; ++l) bias[l][tid] = P.bias[l][tid];
    mlp_stage_output(P.w_out, P.b_out, w5, tid);

    // ---- features: two threads per ray, eight frequencies each (features_body's arithmetic) ----
    {
        const int r = tid >> 1, half = tid & 1;
        const int g = row0 + r;
        mlp_features(g < n ? P.states + 6 * (size_t)g : nullptr, P.radius, P.freqs, half, act[r]);
    }
    __syncthreads();

    for (int l = 0; l < 4; ++l) {
        const u16* wl = P.wpack + pack_offset(l);
        // The weights are the MFMA's A operand and the layer input its B operand, so a lane's D
        // registers hold 4 consecutive output columns of one ray (stored as one 8-byte LDS
        // write): acc[jn][im] is the tile of columns 64 wave + 32 jn .. +31 and rays
        // 32 im .. +31.  Every wave reads its own weight columns (no two waves of a workgroup
        // load the same fragment) and all 128 rays from LDS.  The products and their k order
        // are those of the unswapped product (each D element sums the same 16 products per
        // instruction).
        f32x16 acc[2][4];
        if (l == 0)
            mlp_layer_k<LM_FUSED_KSTEPS0, true>(wl, P.wpack + pack_offset(1), act, wave, lane, acc, wb, wa);
        else
            mlp_layer_k<LM_FUSED_KSTEPS, true>(wl, P.wpack + pack_offset(l < 3 ? l + 1 : l), act, wave, lane, acc, wa, wb);
        __syncthreads();  // every wave has read this layer's input
        // D of register e: column n = 8 (e / 4) + 4 (lane / 32) + e % 4 of the tile, ray
        // lane % 32: registers 4g .. 4g + 3 are columns n0 .. n0 + 3 of one ray
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int n0 = 64 * wave + 32 * j + 8 * g + 4 * (lane >> 5);
                const float4 bv = *reinterpret_cast<const float4*>(&bias[l][n0]);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int m = 32 * i + (lane & 31);
                    const unsigned lo = f2bf2(silu(acc[j][i][4 * g] + bv.x), silu(acc[j][i][4 * g + 1] + bv.y));
                    const unsigned hi = f2bf2(silu(acc[j][i][4 * g + 2] + bv.z), silu(acc[j][i][4 * g + 3] + bv.w));
                    *reinterpret_cast<uint2*>(&act[m][n0]) = make_uint2(lo, hi);
                }
            }
        __syncthreads();
    }

    // ---- output layer (FP32, out_layer_kernel's order) ----
    {
        const int r = 64 * (wave & 1) + lane, o0 = 4 * (wave >> 1);
        const int g = row0 + r;
        const f32x4v s = mlp_output(act[r], w5, o0, lane);
        if (g < n) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (o0 + q < LS_OUT) P.out[(size_t)g * LS_OUT + o0 + q] = s[q];
        }
    }
}

}  // namespace lm
