// Kernels of the learned flow-map surrogate: training (Fourier features, BF16-MFMA GEMMs with
// fused epilogues, an FP32 output layer, loss, split-K weight-gradient reduction, Adam) and a
// frame (RK4 approach to the bounding sphere, MLP inference, RK4 fallback, re-judging).
#include <hip/hip_runtime.h>

#include "device/fields.hpp"
#include "device/loop_fields.hpp"
#include "device/gemm_nt.hpp"
#include "device/gemm_tn.hpp"
#include "device/mlp.hpp"
#include "device/mlp_fused.hpp"
#include "device/surrogate.hpp"
#include "device/train.hpp"
#include "device/train_pass.hpp"
#include "surrogate_kernels.hpp"

namespace LINON_KERNEL_NS {

using lm::u16;

__global__ void __launch_bounds__(256) gemm_kernel(lm::GemmParams P) { lm::gemm_body(P); }
__global__ void __launch_bounds__(256) gemm_nt_kernel(lm::GemmParams P) { lm::gemm_nt_body(P); }
__global__ void __launch_bounds__(256) gemm_tn_kernel(lm::GemmParams P) {
    lm::gemm_tn_body(P, lm::gemm_tn_work((int)blockIdx.x, (int)gridDim.x));
}
// two 128-row workgroups per CU (80 KB of LDS each)
__global__ void __launch_bounds__(256, 2) train_pass_kernel(lm::PassParams P) { lm::train_pass_body(P); }
__global__ void __launch_bounds__(256) grads_kernel(lm::GradParams P) { lm::grads_body(P); }
__global__ void __launch_bounds__(LM_SUM_ROWS) update_kernel(lm::UpdateParams P) { lm::update_body(P); }

__global__ void __launch_bounds__(256) features_kernel(ls::SurrogateIO S) { ls::features_body(S); }
template <bool Transposed>
__global__ void __launch_bounds__(256) mlp_pack_kernel(const float* W, int K, u16* dst) {
    lm::mlp_pack_body<Transposed>(W, K, dst);
}
// two 128-ray workgroups per CU (75 KB of LDS each)
__global__ void __launch_bounds__(256, 2) mlp_infer_kernel(lm::MlpInferParams P) { lm::mlp_infer_body(P); }

template <class F>
__global__ void __launch_bounds__(256) approach_kernel(ls::ApproachParams A) {
    ls::approach_body<F>(A);
}

template <class F>
__global__ void __launch_bounds__(256) flowmap_kernel(ls::FlowmapParams P) {
    ls::flowmap_body<F, false>(P);
}

template <class F>
__global__ void __launch_bounds__(256) flowmap_free_kernel(ls::FlowmapParams P) {
    ls::flowmap_body<F, true>(P);
}

// Uniform entry states: p uniform on the sphere of radius R, pulled inside by up to one step
// (u * inset), q uniform over directions pointing into the sphere (q . p < 0); counter-based
// SplitMix64 stream, so the data set is a function of the seed.
__device__ __forceinline__ float u01(unsigned long long seed, unsigned long long i) {
    unsigned long long z = seed + 0x9E3779B97F4A7C15ull * (i + 1);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (float)(z >> 40) * (1.0f / 16777216.0f);
}
__global__ void __launch_bounds__(256) sample_states_kernel(unsigned long long seed, int n, float radius, float inset,
                                                            float* states) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const unsigned long long b = 6ull * (unsigned long long)i;
    float z1 = 2.0f * u01(seed, b) - 1.0f, ph1 = 6.283185307179586f * u01(seed, b + 1);
    float z2 = 2.0f * u01(seed, b + 2) - 1.0f, ph2 = 6.283185307179586f * u01(seed, b + 3);
    float r = radius - inset * u01(seed, b + 4);
    float s1 = sqrtf(fmaxf(0.0f, 1.0f - z1 * z1)), s2 = sqrtf(fmaxf(0.0f, 1.0f - z2 * z2));
    float px = s1 * cosf(ph1), py = s1 * sinf(ph1), pz = z1;
    float qx = s2 * cosf(ph2), qy = s2 * sinf(ph2), qz = z2;
    if (px * qx + py * qy + pz * qz > 0.0f) {
        qx = -qx;
        qy = -qy;
        qz = -qz;
    }
    float* o = states + 6 * (size_t)i;
    o[0] = r * px; o[1] = r * py; o[2] = r * pz;
    o[3] = qx; o[4] = qy; o[5] = qz;
}

// Appends to a list: every thread of the block calls it (blockDim.x = LS_LIST_BLOCK), those with
// `want` get their slots, in thread order.  One atomic per block: all blocks' go to one address,
// about 9 ns each, which a 1080p frame's kernels with an atomic per wave spent their time on
// (re-judge picks 182 us).
#define LS_LIST_BLOCK 1024
__device__ __forceinline__ int append_slot(bool want, int* count) {
    __shared__ int base[LS_LIST_BLOCK / 64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const unsigned long long lanes = __ballot(want);
    if (lane == 0) base[wave] = __popcll(lanes);
    __syncthreads();
    if (threadIdx.x == 0) {
        int n = 0;
        for (int w = 0; w < LS_LIST_BLOCK / 64; ++w) n += base[w];
        int at = n ? atomicAdd(count, n) : 0;
        for (int w = 0; w < LS_LIST_BLOCK / 64; ++w) {
            const int k = base[w];
            base[w] = at;
            at += k;
        }
    }
    __syncthreads();
    return base[wave] + __popcll(lanes & ((1ull << lane) - 1ull));
}

// Picks roughly one accepted ray in `stride` (hash-spread) for re-judging with RK4.
__global__ void __launch_bounds__(LS_LIST_BLOCK) pick_rejudge_kernel(const int* accepted, int n, const int* n_dev,
                                                                     int stride, unsigned long long seed, int* list,
                                                                     int* count) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int rows = n_dev ? *n_dev : n;
    if ((int)(blockIdx.x * blockDim.x) >= rows) return;  // the whole block
    const bool pick =
        i < rows && accepted[i] && (int)(u01(seed, (unsigned long long)i) * (float)stride) == 0;
    const int slot = append_slot(pick, count);
    if (pick) list[slot] = i;
}

// Network targets of the training set: (exit - base) * scale, per row (point scale for the
// three exit-point values, direction scale for the exit direction); base = the coarse flow map,
// or none (0) when the network predicts the exit itself.
__global__ void __launch_bounds__(256) make_targets_kernel(const float* fine, const float* base, int n,
                                                           float scale_p, float scale_d, float* tgt) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 6 * n) return;
    const int k = t % 6;
    const float b = base ? base[t] : 0.0f;
    tgt[t] = (fine[t] - b) * (k < 3 ? scale_p : scale_d);
}

// Sums of squares of (fine - base) over all rows: acc[0] over the exit-point values, acc[1]
// over the directions (block reduction, one atomic per block and accumulator).
__global__ void __launch_bounds__(256) residual_sumsq_kernel(const float* fine, const float* base, int n, float* acc) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    float sp = 0.0f, sd = 0.0f;
    if (t < n) {
        for (int k = 0; k < 6; ++k) {
            const float d = fine[6 * (size_t)t + k] - (base ? base[6 * (size_t)t + k] : 0.0f);
            (k < 3 ? sp : sd) += d * d;
        }
    }
    __shared__ float red[2][256];
    red[0][threadIdx.x] = sp;
    red[1][threadIdx.x] = sd;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            red[0][threadIdx.x] += red[0][threadIdx.x + s];
            red[1][threadIdx.x] += red[1][threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        atomicAdd(acc, red[0][0]);
        atomicAdd(acc + 1, red[1][0]);
    }
}

// FP32 output layer: out[i][o] = sum_k act[i][k] * W[k][o] + b[o] (bf16 activations, fp32
// weights), one lane per (row, output).
__global__ void __launch_bounds__(256) out_layer_kernel(const u16* act, const float* W, const float* b, int n,
                                                        float* out) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n * LS_OUT) return;
    const int i = t / LS_OUT, o = t % LS_OUT;
    const u16* a = act + (size_t)i * LS_HIDDEN;
    float s = b[o];
    for (int k = 0; k < LS_HIDDEN; ++k) s = __builtin_fmaf(lm::bf2f(a[k]), W[k * LS_OUT + o], s);
    out[(size_t)i * LS_OUT + o] = s;
}

// Exit-point error of every row's prediction (base + output / scale_p) against its RK4 exit.
__global__ void __launch_bounds__(256) errors_kernel(const float* out, const float* target, const float* fine, int n,
                                                     float scale_p, float* err) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float* f = fine + 6 * (size_t)i;
    float pe[3];
    for (int k = 0; k < 3; ++k) pe[k] = f[k] + (out[(size_t)i * LS_OUT + k] - target[6 * (size_t)i + k]) / scale_p;
    err[i] = lm::exit_error(pe[0], pe[1], pe[2], f);
}

// The BF16 copy [N][K] of a hidden layer's weights W [K][N], N = 256.
__global__ void __launch_bounds__(256) transpose_kernel(const float* W, int K, u16* wt) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= K * LS_HIDDEN) return;
    const int n = t / K, k = t % K;
    wt[t] = lm::f2bf(W[(size_t)k * LS_HIDDEN + n]);
}

// Sums split-K partials: out[j] = sum_s part[s][j].
__global__ void __launch_bounds__(256) reduce_partials_kernel(const float* part, int splits, int n, float* out) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    float s = 0.0f;
    for (int k = 0; k < splits; ++k) s += part[(size_t)k * n + j];
    out[j] = s;
}

// Surrogate verdict per entered ray: accept (write the exit point to the mapping) when the
// confidence reaches the threshold; otherwise queue the ray for RK4.  The exit point is the
// base (coarse flow map, or 0) plus the output over the point scale.
__global__ void __launch_bounds__(LS_LIST_BLOCK) accept_kernel(const float* out, const float* base,
                                                               const int* texel_of, int n, const int* n_dev,
                                                               float scale_p, float conf_threshold, float* mapping,
                                                               float* pred_exit, int* fallback, int* n_fallback,
                                                               int* accepted) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int rows = n_dev ? *n_dev : n;
    if ((int)(blockIdx.x * blockDim.x) >= rows) return;  // the whole block
    bool accept = true;
    if (i < rows) {
        const float* o = out + (size_t)i * LS_OUT;
        const float conf = 1.0f / (1.0f + __expf(-o[6]));
        const float inv = 1.0f / scale_p;
        const float* b = base ? base + 6 * (size_t)i : nullptr;
        const float px = (b ? b[0] : 0.0f) + o[0] * inv, py = (b ? b[1] : 0.0f) + o[1] * inv,
                    pz = (b ? b[2] : 0.0f) + o[2] * inv;
        pred_exit[3 * (size_t)i] = px;
        pred_exit[3 * (size_t)i + 1] = py;
        pred_exit[3 * (size_t)i + 2] = pz;
        accept = conf >= conf_threshold;
        accepted[i] = accept ? 1 : 0;
        if (accept) reinterpret_cast<float4*>(mapping)[texel_of[i]] = make_float4(px, py, pz, 1.0f);
    }
    const int slot = append_slot(!accept, n_fallback);
    if (!accept) fallback[slot] = i;
}

// Rays re-judged by RK4 or sent to RK4: write the RK4 exit into the mapping; for re-judged
// rays also record the surrogate's error against the RK4 exit (exit_error).
__global__ void __launch_bounds__(256) apply_rk4_kernel(const int* list, int n, const int* n_dev, const float* exits,
                                                        const int* texel_of, const float* pred_exit, float* mapping,
                                                        float* err_out, int write_mapping) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (n_dev ? *n_dev : n)) return;
    const int r = list[i];
    const float* e = exits + 6 * (size_t)r;
    if (err_out)
        err_out[i] = lm::exit_error(pred_exit[3 * (size_t)r], pred_exit[3 * (size_t)r + 1], pred_exit[3 * (size_t)r + 2], e);
    if (write_mapping) reinterpret_cast<float4*>(mapping)[texel_of[r]] = make_float4(e[0], e[1], e[2], 1.0f);
}

// Accepted rays whose Lyapunov exponent (from the surrogate's own mapping) is above the
// threshold are queued for RK4 as well, and no longer count as accepted.
__global__ void __launch_bounds__(LS_LIST_BLOCK) lyapunov_gate_kernel(int* accepted, const int* texel_of, int n,
                                                                      const int* n_dev, const float* lyap,
                                                                      float threshold, int* list, int* count) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int rows = n_dev ? *n_dev : n;
    if ((int)(blockIdx.x * blockDim.x) >= rows) return;  // the whole block
    const bool gate = i < rows && accepted[i] && lyap[texel_of[i]] > threshold;
    const int slot = append_slot(gate, count);
    if (gate) {
        accepted[i] = 0;
        list[slot] = i;
    }
}

// Per texel: 1 where the frame kept the surrogate's exit (mask cleared beforehand).
__global__ void __launch_bounds__(256) accepted_mask_kernel(const int* accepted, const int* texel_of, int n,
                                                            const int* n_dev, unsigned char* mask) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < (n_dev ? *n_dev : n) && accepted[i]) mask[texel_of[i]] = 1;
}

__global__ void __launch_bounds__(256) fill_u8_kernel(unsigned char* p, int n, unsigned char value) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

__global__ void __launch_bounds__(256) fill_i32_kernel(int* p, int n, int value) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

// ---- launchers ------------------------------------------------------------------------------
hipError_t sg_gemm(const lm::GemmParams& P, int splits, hipStream_t s) {
    void* args[] = {const_cast<lm::GemmParams*>(&P)};
    if (splits == 1 && lm::gemm_nt_applies(P)) {  // the forward layout: 128 x 128 tiles, 16-B loads
        dim3 grid((P.M + LM_NT_BM - 1) / LM_NT_BM, P.N / LM_NT_BN, 1);
        return hipLaunchKernel((const void*)&gemm_nt_kernel, grid, dim3(256), args, 0, s);
    }
    if (lm::gemm_tn_applies(P))  // the weight gradients' layout: register-transposed 128 x 128 tiles
        return hipLaunchKernel((const void*)&gemm_tn_kernel, dim3(lm::gemm_tn_tiles(P) * splits), dim3(256), args, 0, s);
    dim3 grid((P.M + LM_BM - 1) / LM_BM, (P.N + LM_BN - 1) / LM_BN, splits);
    return hipLaunchKernel((const void*)&gemm_kernel, grid, dim3(256), args, 0, s);
}

#define LS_GRID(n) dim3(((n) + 255) / 256), dim3(256)
#define LS_LIST_GRID(n) dim3(((n) + LS_LIST_BLOCK - 1) / LS_LIST_BLOCK), dim3(LS_LIST_BLOCK)

hipError_t sg_mlp_pack(const float* W, int K, u16* dst, bool transposed, hipStream_t s) {
    if (transposed)
        hipLaunchKernelGGL(mlp_pack_kernel<true>, LS_GRID((K / 16) * 8 * 64), 0, s, W, K, dst);
    else
        hipLaunchKernelGGL(mlp_pack_kernel<false>, LS_GRID((K / 16) * 8 * 64), 0, s, W, K, dst);
    return hipGetLastError();
}
hipError_t sg_mlp_infer(const lm::MlpInferParams& P, hipStream_t s) {
    if (P.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(mlp_infer_kernel, dim3((P.n + LM_FUSED_ROWS - 1) / LM_FUSED_ROWS), dim3(256), 0, s, P);
    return hipGetLastError();
}
hipError_t sg_features(const ls::SurrogateIO& S, hipStream_t s) {
    hipLaunchKernelGGL(features_kernel, LS_GRID(S.n), 0, s, S);
    return hipGetLastError();
}
hipError_t sg_make_targets(const float* fine, const float* base, int n, float scale_p, float scale_d, float* tgt,
                           hipStream_t s) {
    hipLaunchKernelGGL(make_targets_kernel, LS_GRID(6 * n), 0, s, fine, base, n, scale_p, scale_d, tgt);
    return hipGetLastError();
}
hipError_t sg_residual_sumsq(const float* fine, const float* base, int n, float* acc, hipStream_t s) {
    hipLaunchKernelGGL(residual_sumsq_kernel, LS_GRID(n), 0, s, fine, base, n, acc);
    return hipGetLastError();
}
hipError_t sg_train_pass(const lm::PassParams& P, hipStream_t s) {
    hipLaunchKernelGGL(train_pass_kernel, dim3((P.rows + LM_FUSED_ROWS - 1) / LM_FUSED_ROWS), dim3(256), 0, s, P);
    return hipGetLastError();
}
hipError_t sg_transpose(const float* W, int K, u16* wt, hipStream_t s) {
    hipLaunchKernelGGL(transpose_kernel, LS_GRID(K * LS_HIDDEN), 0, s, W, K, wt);
    return hipGetLastError();
}
hipError_t sg_errors(const float* out, const float* target, const float* fine, int n, float scale_p, float* err,
                     hipStream_t s) {
    hipLaunchKernelGGL(errors_kernel, LS_GRID(n), 0, s, out, target, fine, n, scale_p, err);
    return hipGetLastError();
}
hipError_t sg_out_layer(const u16* act, const float* W, const float* b, int n, float* out, hipStream_t s) {
    hipLaunchKernelGGL(out_layer_kernel, LS_GRID(n * LS_OUT), 0, s, act, W, b, n, out);
    return hipGetLastError();
}
hipError_t sg_reduce(const float* part, int splits, int n, float* out, hipStream_t s) {
    hipLaunchKernelGGL(reduce_partials_kernel, LS_GRID(n), 0, s, part, splits, n, out);
    return hipGetLastError();
}
hipError_t sg_grads(const lm::GradParams& P, hipStream_t s) {
    for (const lm::GemmParams& dw : P.dw)  // the tiles read whole steps only, and know no other loop
        if (!lm::gemm_tn_applies(dw)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(grads_kernel, dim3(lm::grads_sum_blocks() + lm::grads_tiles(P)), dim3(256), 0, s, P);
    return hipGetLastError();
}
hipError_t sg_update(const lm::UpdateParams& P, hipStream_t s) {
    hipLaunchKernelGGL(update_kernel, dim3(lm::update_blocks(P)), dim3(LM_SUM_ROWS), 0, s, P);
    return hipGetLastError();
}
hipError_t sg_accept(const float* out, const float* base, const int* texel_of, int n, const int* n_dev, float scale_p,
                     float thr, float* mapping, float* pred_exit, int* fallback, int* n_fallback, int* accepted,
                     hipStream_t s) {
    hipLaunchKernelGGL(accept_kernel, LS_LIST_GRID(n), 0, s, out, base, texel_of, n, n_dev, scale_p, thr, mapping,
                       pred_exit, fallback, n_fallback, accepted);
    return hipGetLastError();
}
hipError_t sg_apply_rk4(const int* list, int n, const int* n_dev, const float* exits, const int* texel_of,
                        const float* pred_exit, float* mapping, float* err_out, int write_mapping, hipStream_t s) {
    hipLaunchKernelGGL(apply_rk4_kernel, LS_GRID(n), 0, s, list, n, n_dev, exits, texel_of, pred_exit, mapping, err_out,
                       write_mapping);
    return hipGetLastError();
}
hipError_t sg_accepted_mask(const int* accepted, const int* texel_of, int n, const int* n_dev, int npx,
                            unsigned char* mask, hipStream_t s) {
    hipLaunchKernelGGL(fill_u8_kernel, LS_GRID(npx), 0, s, mask, npx, (unsigned char)0);
    if (n > 0) hipLaunchKernelGGL(accepted_mask_kernel, LS_GRID(n), 0, s, accepted, texel_of, n, n_dev, mask);
    return hipGetLastError();
}
hipError_t sg_lyapunov_gate(int* accepted, const int* texel_of, int n, const int* n_dev, const float* lyap, float thr,
                            int* list, int* count, hipStream_t s) {
    hipLaunchKernelGGL(lyapunov_gate_kernel, LS_LIST_GRID(n), 0, s, accepted, texel_of, n, n_dev, lyap, thr, list, count);
    return hipGetLastError();
}
hipError_t sg_sample_states(unsigned long long seed, int n, float radius, float inset, float* states, hipStream_t s) {
    hipLaunchKernelGGL(sample_states_kernel, LS_GRID(n), 0, s, seed, n, radius, inset, states);
    return hipGetLastError();
}
hipError_t sg_pick_rejudge(const int* accepted, int n, const int* n_dev, int stride, unsigned long long seed, int* list,
                           int* count, hipStream_t s) {
    hipLaunchKernelGGL(pick_rejudge_kernel, LS_LIST_GRID(n), 0, s, accepted, n, n_dev, stride, seed, list, count);
    return hipGetLastError();
}
hipError_t sg_fill_i32(int* p, int n, int value, hipStream_t s) {
    hipLaunchKernelGGL(fill_i32_kernel, LS_GRID(n), 0, s, p, n, value);
    return hipGetLastError();
}

#define LS_FIELD_CASES(KERNEL)                                               \
    case 17: return (const void*)&KERNEL<lw::FieldSwirl>;                    \
    case 19: return (const void*)&KERNEL<lw::FieldHotAir>;                   \
    case 20: return (const void*)&KERNEL<lw::FieldWarp>;                     \
    case LINON_KERNEL_HOT_AIR_FAITHFUL_ROOT:                                 \
        return (const void*)&KERNEL<lw::FieldHotAirFaithfulRoot>;            \
    case 3: return (const void*)&KERNEL<lw::FieldMirageSphericalSigmoid>;    \
    case 16: return (const void*)&KERNEL<lw::FieldIdentity>;                 \
    default: return nullptr;
#define LS_LENS_CASES(KERNEL)                                                \
    case 18: return (const void*)&KERNEL<lw::FieldLens>;                     \
    case LINON_KERNEL_LENS_RECIP:                                            \
        return (const void*)&KERNEL<lw::FieldLensRecip>;

static const void* approach_for(int field) {
    switch (field) { LS_LENS_CASES(approach_kernel) LS_FIELD_CASES(approach_kernel) }
}
static const void* flowmap_for(int field) {
    switch (field) { LS_LENS_CASES(flowmap_kernel) LS_FIELD_CASES(flowmap_kernel) }
}
// Fixed steps in the loop without a mesh: faster from one ray to 400,000 (ray_advance_free's
// figures).  Not the lens, whose step is mostly its field's own branches: with the outward test at
// every step 844,000 rays took 9.12 ms so and 8.97 in the general loop, 3,000 rays 1.03-1.20 and
// 1.16 ms a call.
static const void* flowmap_free_for(int field) {
    switch (field) { LS_FIELD_CASES(flowmap_free_kernel) }
}

bool sg_field_supported(int field) { return approach_for(field) != nullptr; }

hipError_t sg_approach(int field, const ls::ApproachParams& A, hipStream_t s) {
    const void* fn = approach_for(field);
    if (!fn) return hipErrorInvalidDeviceFunction;
    const int tiles = A.tiles_x * ((A.cam.height + LINON_TILE - 1) / LINON_TILE);
    void* args[] = {const_cast<ls::ApproachParams*>(&A)};
    return hipLaunchKernel(fn, dim3((tiles + 3) / 4), dim3(256), args, 0, s);
}
hipError_t sg_flowmap(int field, const ls::FlowmapParams& P, hipStream_t s) {
    // adaptive steps (a caller's integrator) need the general loop
    const void* fn = P.step.adaptive ? nullptr : flowmap_free_for(field);
    if (!fn) fn = flowmap_for(field);
    if (!fn) return hipErrorInvalidDeviceFunction;
    if (P.n <= 0) return hipSuccess;
    void* args[] = {const_cast<ls::FlowmapParams*>(&P)};
    return hipLaunchKernel(fn, dim3((P.n + 255) / 256), dim3(256), args, 0, s);
}

}  // namespace LINON_KERNEL_NS
