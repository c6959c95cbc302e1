// Forward and backward pass of one training step for 128 rows of the mini-batch in one workgroup:
// gather, Fourier features, four hidden layers, FP32 output layer, loss, and the chain of dZ back
// to the first layer.  One launch a step replaces gather, features, four forward GEMMs, output
// layer, loss, output-layer backward and three dX GEMMs.
//
//   * The layer products are mlp_layer_k's (mlp_fused.hpp): 4 waves, each all 128 rows by 64
//     columns, the layer input in LDS, the weights prepacked in fragment order; backward, the
//     input is dZ and the packed operand W^T.
//   * What the weight gradients need leaves as bf16 rows: the features, the four activations and
//     the four dZ, each copied from the LDS tile in 16-byte pieces while the next layer's product
//     reads the same tile.
//   * The pre-activations z stay FP32.  The last layer's never leaves its accumulators; the other
//     three go to scratch in the accumulators' own order (each thread reads back what it wrote, 16
//     bytes a lane, 1 KB a wave), not as a row-major matrix.
// What bounds it: at 65536 rows, 290 MB of bf16 rows and 400 MB of z to and from memory, and the
// SiLU and its derivative (an exponential and a reciprocal each, quarter rate) beside the MFMAs.
// 174 us there; the launches it replaces took 895 (600 of them the dX products on 2-byte loads).
// Rows and z move nontemporally: as ordinary stores they push one another and the weights out of the
// caches (185 us; the rows alone 176 and z alone 172, but then the gradients' launch that reads the
// rows takes 112 us and not 106).
// The weights of a layer are first read at its start: read under the layer before, as inference
// does, they cost 190 bytes of spills more and the pass took 217 us for 189.
//
// The arithmetic is that of the kernels it replaces (features_body, gemm_body's k order,
// out_layer_kernel's and loss_kernel's expressions): the same bits.
#pragma once
#include "mlp_fused.hpp"
#include "train.hpp"

namespace lm {

struct PassParams {
    // the training set and the mini-batch drawn from it
    const float* states;    // [n_data][6]
    const float* targets;   // [n_data][6] network targets
    const float* fine;      // [n_data][6] RK4 exits
    int n_data;
    unsigned long long seed;
    int step;
    int rows;               // mini-batch rows
    // the network
    float radius;
    const float* freqs;     // [LS_FREQS]
    const u16* wpack;       // LM_PACK_TOTAL forward fragments
    const u16* bpack;       // 3 * LM_PACK_LAYER backward fragments of layers 1..3
    const float* bias[4];
    const float* w_out;     // [256][LS_OUT]
    const float* b_out;
    // the loss
    float scale_p, tol, conf_weight;
    float* loss;            // optional: mean loss is added
    // what the gradients read
    u16* feat;              // [rows][LS_FEATS_PAD]
    u16* act[4];            // [rows][256] outputs of the hidden layers
    u16* dz[4];             // [rows][256]
    float* dout;            // [rows][LS_OUT]
    float* z;               // [3][row tiles][32][256] float4: z of layers 0..2 in register order
};

// Exit-point error of a prediction against the RK4 exit, as the parity tests measure it:
// max over x, y, z of |pred - exit| / max(1, |exit|).
__device__ __forceinline__ float exit_error(float px, float py, float pz, const float* e) {
    const float ex = fabsf(px - e[0]) / fmaxf(1.0f, fabsf(e[0]));
    const float ey = fabsf(py - e[1]) / fmaxf(1.0f, fabsf(e[1]));
    const float ez = fabsf(pz - e[2]) / fmaxf(1.0f, fabsf(e[2]));
    return fmaxf(ex, fmaxf(ey, ez));
}

// The LDS tile's first `chunks` 16-byte pieces of each row to out [rows][8 chunks] bf16.
template <int Chunks>
__device__ __forceinline__ void tile_out(const u16 (*tile)[LM_FUSED_LDA], int row0, int n, u16* out) {
#pragma unroll 4
    for (int i = threadIdx.x; i < LM_FUSED_ROWS * Chunks; i += 256) {
        const int r = i / Chunks, c = i % Chunks;
        if (row0 + r < n)
            __builtin_nontemporal_store(*reinterpret_cast<const u32x4v*>(&tile[r][c * 8]),
                                        reinterpret_cast<u32x4v*>(out + ((size_t)(row0 + r) * Chunks + c) * 8));
    }
}

__device__ __forceinline__ void train_pass_body(const PassParams& P) {
    __shared__ __attribute__((aligned(16))) u16 tile[LM_FUSED_ROWS][LM_FUSED_LDA];
    __shared__ __attribute__((aligned(16))) float w5[8][LM_FUSED_W5];   // the 7 outputs and a zero
    __shared__ __attribute__((aligned(16))) float d5[LM_FUSED_ROWS][8]; // dOut of each row and a zero
    __shared__ float wave_loss[4];
    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int row0 = blockIdx.x * LM_FUSED_ROWS;
    const int n = P.rows;
    mlp_stage_output(P.w_out, P.b_out, w5, tid);

    // ---- gather and features: two threads per row, eight frequencies each ----
    const int r = tid >> 1, half = tid & 1;
    const bool in = row0 + r < n;
    size_t src = 0;  // row of the training set: a counter-based hash of (seed, step, i)
    if (in) {
        unsigned long long h = P.seed + 0x9E3779B97F4A7C15ull * ((unsigned long long)P.step * (unsigned long long)n +
                                                                 (unsigned long long)(row0 + r) + 1);
        h = (h ^ (h >> 30)) * 0xBF58476D1CE4E5B9ull;
        h = (h ^ (h >> 27)) * 0x94D049BB133111EBull;
        h ^= h >> 31;
        src = (size_t)(h % (unsigned long long)P.n_data);
    }
    mlp_features(in ? P.states + 6 * src : nullptr, P.radius, P.freqs, half, tile[r]);
    __syncthreads();

    f32x16 acc[2][4];
    // this thread's z scratch of layer l: 32 float4, 256 threads apart
    const size_t tiles = gridDim.x;
    auto zat = [&](int l) {
        return reinterpret_cast<f32x4v*>(P.z) + (((size_t)l * tiles + blockIdx.x) * 32) * 256 + tid;
    };
    const int nl = 64 * wave + 4 * (lane >> 5);  // this lane's columns are nl + 32 j + 8 g .. +3, its rows 32 i + lane % 32

    // ---- forward ----
    // bias, SiLU, and the pre-activations to scratch but for the last layer's, in one straight piece
    // each (a test at every store left pieces of 26 instructions whose exponentials had nothing to
    // overlap with)
    auto epilogue = [&](const float* bias, f32x4v* z, auto keep) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int n0 = nl + 32 * j + 8 * g;
                const float4 bv = *reinterpret_cast<const float4*>(bias + n0);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    f32x16& a = acc[j][i];
                    a[4 * g] += bv.x;
                    a[4 * g + 1] += bv.y;
                    a[4 * g + 2] += bv.z;
                    a[4 * g + 3] += bv.w;
                    if constexpr (!decltype(keep)::value)
                        __builtin_nontemporal_store(f32x4v{a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]},
                                                    &z[((j * 4 + g) * 4 + i) * 256]);
                    const unsigned lo = f2bf2(silu(a[4 * g]), silu(a[4 * g + 1]));
                    const unsigned hi = f2bf2(silu(a[4 * g + 2]), silu(a[4 * g + 3]));
                    *reinterpret_cast<uint2*>(&tile[32 * i + (lane & 31)][n0]) = make_uint2(lo, hi);
                }
            }
        __syncthreads();
    };
    u32x4v wa[2][2], wb[2][2];
#pragma nounroll
    for (int l = 0; l < 3; ++l) {
        const u16* wl = P.wpack + pack_offset(l);
        mlp_load_pair(wl, 0, wave, lane, wa);
        if (l == 0) {
            tile_out<LS_FEATS_PAD / 8>(tile, row0, n, P.feat);
            mlp_layer_k<LM_FUSED_KSTEPS0, false>(wl, nullptr, tile, wave, lane, acc, wa, wb);
        } else {
            tile_out<LS_HIDDEN / 8>(tile, row0, n, P.act[l - 1]);
            mlp_layer_k<LM_FUSED_KSTEPS, false>(wl, nullptr, tile, wave, lane, acc, wa, wb);
        }
        __syncthreads();  // every wave has read this layer's input
        epilogue(P.bias[l], zat(l), IntType<0>{});
    }
    mlp_load_pair(P.wpack + pack_offset(3), 0, wave, lane, wa);
    tile_out<LS_HIDDEN / 8>(tile, row0, n, P.act[2]);
    mlp_layer_k<LM_FUSED_KSTEPS, false>(P.wpack + pack_offset(3), nullptr, tile, wave, lane, acc, wa, wb);
    __syncthreads();
    epilogue(P.bias[3], nullptr, IntType<1>{});

    // ---- output layer and loss: two threads per row (outputs 0..3 and 4..6); z of the last
    // layer stays in acc ----
    tile_out<LS_HIDDEN / 8>(tile, row0, n, P.act[3]);
    float loss = 0.0f;
    {
        const int ray = 64 * (wave & 1) + lane, oq = 4 * (wave >> 1);
        *reinterpret_cast<f32x4v*>(&d5[ray][oq]) = mlp_output(tile[ray], w5, oq, lane);
        __syncthreads();
        const int o0 = 4 * half;
        const float4 sv = *reinterpret_cast<const float4*>(&d5[r][o0]);
        const float s[4] = {sv.x, sv.y, sv.z, sv.w};
        float d[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (in) {
            const float* y = P.targets + 6 * src;
            const float* f = P.fine + 6 * src;
            float pe[3] = {0.0f, 0.0f, 0.0f};
            const int nk = half ? 2 : 4;
            for (int q = 0; q < nk; ++q) {  // the six regression outputs
                const int k = o0 + q;
                const float e = s[q] - y[k];
                loss += e * e / 6.0f;
                d[q] = 2.0f * e / (6.0f * n);
                if (k < 3) pe[q] = f[k] + e / P.scale_p;  // the prediction: exit + (output - target) / scale
            }
            float label = half ? 0.0f : (exit_error(pe[0], pe[1], pe[2], f) <= P.tol ? 1.0f : 0.0f);
            label = __shfl(label, lane & ~1);
            if (half) {  // the confidence: logistic loss against [error <= tol]
                const float c = s[2];
                const float p = 1.0f / (1.0f + __expf(-c));
                loss += P.conf_weight * (fmaxf(c, 0.0f) - c * label + log1pf(__expf(-fabsf(c))));
                d[2] = P.conf_weight * (p - label) / n;
            }
            float* o = P.dout + (size_t)(row0 + r) * LS_OUT + o0;
            for (int q = 0; q < (half ? 3 : 4); ++q) o[q] = d[q];
        }
        *reinterpret_cast<float4*>(&d5[r][o0]) = make_float4(d[0], d[1], d[2], d[3]);
    }
    if (P.loss) {
        for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off, 64);
        if (lane == 0) wave_loss[wave] = loss;
    }
    __syncthreads();  // dOut is complete, and every wave has read the last activations
    if (P.loss && tid == 0) atomicAdd(P.loss, (((wave_loss[0] + wave_loss[1]) + wave_loss[2]) + wave_loss[3]) / n);

    // ---- dZ of the last layer: (sum over o of dOut W) * silu'(z) ----
    {
        float4 da[4], db[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            da[i] = *reinterpret_cast<const float4*>(&d5[32 * i + (lane & 31)][0]);
            db[i] = *reinterpret_cast<const float4*>(&d5[32 * i + (lane & 31)][4]);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int n0 = nl + 32 * j + 8 * g;
                float4 w[LS_OUT];
#pragma unroll
                for (int o = 0; o < LS_OUT; ++o) w[o] = *reinterpret_cast<const float4*>(&w5[o][n0]);
                float t[4][4];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    auto wc = [&](int o) { return c == 0 ? w[o].x : c == 1 ? w[o].y : c == 2 ? w[o].z : w[o].w; };
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        float s = __builtin_fmaf(da[i].x, wc(0), 0.0f);
                        s = __builtin_fmaf(da[i].y, wc(1), s);
                        s = __builtin_fmaf(da[i].z, wc(2), s);
                        s = __builtin_fmaf(da[i].w, wc(3), s);
                        s = __builtin_fmaf(db[i].x, wc(4), s);
                        s = __builtin_fmaf(db[i].y, wc(5), s);
                        s = __builtin_fmaf(db[i].z, wc(6), s);
                        t[i][c] = s * silu_grad(acc[j][i][4 * g + c]);
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    *reinterpret_cast<uint2*>(&tile[32 * i + (lane & 31)][n0]) =
                        make_uint2(f2bf2(t[i][0], t[i][1]), f2bf2(t[i][2], t[i][3]));
            }
        __syncthreads();
    }

    // ---- dZ of layer l - 1 = (dZ W^T) * silu'(z_{l-1}) ----
#pragma nounroll
    for (int l = 3; l > 0; --l) {
        const u16* wl = P.bpack + (size_t)(l - 1) * LM_PACK_LAYER;
        mlp_load_pair(wl, 0, wave, lane, wa);
        tile_out<LS_HIDDEN / 8>(tile, row0, n, P.dz[l]);
        mlp_layer_k<LM_FUSED_KSTEPS, false>(wl, nullptr, tile, wave, lane, acc, wa, wb);
        __syncthreads();
        const f32x4v* z = zat(l - 1);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int n0 = nl + 32 * j + 8 * g;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const f32x4v zv = __builtin_nontemporal_load(&z[((j * 4 + g) * 4 + i) * 256]);
                    const f32x16& a = acc[j][i];
                    const unsigned lo = f2bf2(a[4 * g] * silu_grad(zv.x), a[4 * g + 1] * silu_grad(zv.y));
                    const unsigned hi = f2bf2(a[4 * g + 2] * silu_grad(zv.z), a[4 * g + 3] * silu_grad(zv.w));
                    *reinterpret_cast<uint2*>(&tile[32 * i + (lane & 31)][n0]) = make_uint2(lo, hi);
                }
            }
        __syncthreads();
    }
    tile_out<LS_HIDDEN / 8>(tile, row0, n, P.dz[0]);
}

}  // namespace lm
