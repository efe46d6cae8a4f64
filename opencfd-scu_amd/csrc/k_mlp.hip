// k_mlp.hip - learned hybrid sensor (gfx950).
//
// A small MLP (24 -> 32 -> 32 -> 1, GELU, sigmoid) stands beside the
// hybrid_auto style-2 selector (Set_Scheme_HybridAuto / Comput_Scheme_point_
// Jameson, src/OCFD_Schemes_hybrid_auto.cu:21-68, 611-703).  It has no
// counterpart in the reference.
//
//   k_mlp_sensor  features of a node (8 per direction, FP32) -> BF16 -> two
//                 16x16x16 BF16 MFMA layers per wave of 64 nodes (FP32
//                 accumulation), GELU, the output dot product with a
//                 16-lane reduction, sigmoid; the flag is the plain kp where
//                 the probability lies in [lo, hi] (low confidence), 1 (UP7)
//                 below lo and max(kp, 2) above hi.  The plain dp is
//                 computed in the same kernel (mlp_dev.h holds these steps,
//                 which the x sweep of the first RK stage runs as well).
//                 Flags are written once per step, at the first RK stage,
//                 like the plain sensor's.
//   k_mlp_collect features and plain labels (kp > 1) of the nodes of a
//                 sub-lattice, for training.
//   k_mlp_grad / k_mlp_update   training in FP32 (FP32 MFMA): forward,
//                 backward and partial gradient sums per wave, then the sum
//                 of the partials and the Adam update (no atomics: neither
//                 depends on scheduling).
//
// Parameters (1889 floats): W1 [32][24], b1 [32], W2 [32][32], b2 [32],
// W3 [32], b3.
#include <hip/hip_runtime.h>

#include "mlp_dev.h"
#include "ocfd_dev.h"
#include "ocfd_kernels.h"

namespace {

using namespace mlp;
static_assert(OB3 + 1 == MLP_NPARAM, "parameter layout");

// ---------------------------------------------------------------------------
// Inference
// ---------------------------------------------------------------------------
// plane = 0: every node with interior indices >= -1 (the whole pass);
// plane = 1: the nodes (i >= 0, j = -1, k >= 0), whose flag only the y sweep
// reads (face -1/2); plane = 2: the nodes (i >= 0, j >= 0, k = -1) for the z
// sweep.  The x sweep of the first RK stage computes the other nodes itself
// (k_sweep_x with LEARN), and planes 1 and 2 complete it.
// The lane fragments of the weights in the layout lane_weights_packed reads
// (one wave).
__global__ void __launch_bounds__(64) k_mlp_pack(const float* __restrict__ P, float* __restrict__ pk) {
    Lane L;
    lane_weights(P, threadIdx.x, L);
    pack_lane(L, threadIdx.x, pk);
}

// P = the packed weights (k_mlp_pack).
template <typename S>
__global__ void __launch_bounds__(256) k_mlp_sensor(FeatIn<S> F, const float* __restrict__ P, double i1, double i2,
                                                    float lo, float hi, int8_t* fx, int8_t* fy, int8_t* fz,
                                                    float* prob_out, int plane) {
    __shared__ unsigned short sX[4][64 * LS];
    const Geo& g = F.g;
    const int lane = threadIdx.x, wv = threadIdx.y;
    Lane L;
    lane_weights_packed(P, lane, L);
    const Blk B = xcd_block();
    int i, j, k;
    bool own;
    if (plane == 0) {
        i = B.x * 64 + lane - 1; j = B.y * 4 + wv - 1; k = B.z - 1;
        own = i < g.nx && j < g.ny;
    } else if (plane == 1) {
        i = B.x * 64 + lane; j = -1; k = B.y * 4 + wv;
        own = i < g.nx && k < g.nz;
    } else {
        i = B.x * 64 + lane; j = B.y * 4 + wv; k = -1;
        own = i < g.nx && j < g.ny;
    }
    const int ic = min(i, g.nx - 1), jc = min(j, g.ny - 1), kc = min(k, g.nz - 1);
    float f[NF];
    features(F, ic, jc, kc, f);
    const float prob = wave_prob(f, sX[wv], L, lane);
    if (!own) return;
    const long long q = gidx(g, i, j, k);
    const int fl = flag_rule(prob, jameson_kp(F, q, i1, i2), lo, hi);
    if (j >= 0 && k >= 0) fx[q] = (int8_t)fl;
    if (i >= 0 && k >= 0) fy[q] = (int8_t)fl;
    if (i >= 0 && j >= 0) fz[q] = (int8_t)fl;
    if (prob_out) prob_out[q] = prob;
}

// ---------------------------------------------------------------------------
// Training data and training
// ---------------------------------------------------------------------------
template <typename S>
__global__ void __launch_bounds__(256) k_mlp_collect(FeatIn<S> F, int stride, int nlx, int nly, int nlz, double i1,
                                                     double i2, float* X, float* y) {
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long n = (long long)nlx * nly * nlz;
    if (t >= n) return;
    const int a = (int)(t % nlx), b = (int)((t / nlx) % nly), c = (int)(t / ((long long)nlx * nly));
    const int i = a * stride, j = b * stride, k = c * stride;
    float f[NF];
    features(F, i, j, k, f);
#pragma unroll
    for (int e = 0; e < NF; e++) X[t * NF + e] = f[e];
    y[t] = jameson_kp(F, gidx(F.g, i, j, k), i1, i2) > 1 ? 1.f : 0.f;
}

// ---------------------------------------------------------------------------
// Training: a wave takes tiles of 32 samples.  All five contractions of a
// tile run on the FP32 matrix instruction v_mfma_f32_32x32x2_f32 (FP32
// products and sums): Z1 = W1 X^T, Z2 = W2 A1, dA1 = W2^T dZ2, dW1 += dZ1 X,
// dW2 += dZ2 A1^T.  A lane l of the instruction holds A[l%32][l/32],
// B[l/32][l%32] and D[unit(r, l/32)][l%32], r = 0..15, unit(r, h) = 8 (r/4) +
// 4 h + r%4.  With samples as columns, register r of one layer's output is
// step r's B operand of the next when the weights are fed in the same unit
// order, so the forward and the backward pass stay in registers; the two
// weight gradients contract over samples and read their operands back from
// LDS tiles (pitch 33: no bank conflicts).  A wave keeps its gradient sums in
// registers over its tiles and writes one partial vector; k_mlp_update adds
// the partials in wave order and applies Adam.  No atomics: a seed fixes the
// result.
//
// Bound by latency, not by work (a batch of 4096 is 0.05 GFLOP): 128 waves of
// one tile instead of one thread per sample and per parameter.  An epoch of
// 65536 samples in batches of 4096, the shuffle on the host included: 33.8 ->
// 0.47 ms (the sum over the samples was one thread per parameter).
// ---------------------------------------------------------------------------
typedef float v16f __attribute__((ext_vector_type(16)));
constexpr int TS = 32;              // samples per tile
constexpr int TP = 33;              // LDS pitch of a 32 x 32 tile
constexpr int PART = MLP_NPARAM + 1;  // a wave's partial: the parameters' gradient sums, then the loss sum
constexpr int MAX_PART = 1024;      // waves (partials) of one batch at most
constexpr int UPD_SLICES = 16;      // partial sums taken beside each other in k_mlp_update

int mlp_waves(int nb) {  // nb >= 1, up to the largest int
    const int t = (nb - 1) / TS + 1;
    return t < MAX_PART ? t : MAX_PART;
}

// GELU and its derivative from one tanh.
__device__ __forceinline__ void gelu_both(float x, float& g, float& dg) {
    const float t = tanhf(0.7978845608028654f * (x + 0.044715f * x * x * x));
    g = 0.5f * x * (1.0f + t);
    dg = 0.5f * (1.0f + t) + 0.5f * x * (1.0f - t * t) * 0.7978845608028654f * (1.0f + 3.0f * 0.044715f * x * x);
}

// GRAD: partial gradient sums of the samples (idx[0..nb), or rows 0..nb) into
// part[gridDim.x][PART]; else only the probabilities into prob.
template <bool GRAD>
__global__ void __launch_bounds__(64) k_mlp_grad(const float* __restrict__ P, const float* __restrict__ X,
                                                 const float* __restrict__ y, const int* __restrict__ idx, int nb,
                                                 float wpos, float* __restrict__ part, float* __restrict__ prob) {
    __shared__ float sX[GRAD ? TS * TP : 1], sD1[GRAD ? TS * TP : 1], sA1[GRAD ? TS * TP : 1],
        sD2[GRAD ? TS * TP : 1], sG3[GRAD ? TS * TP : 1];
    const int lane = threadIdx.x, col = lane & 31, half = lane >> 5;
    auto unit = [&](int r) { return 8 * (r >> 2) + 4 * half + (r & 3); };
    float w1[12], w2[16], w2t[16], w3[16];
    v16f b1, b2;
#pragma unroll
    for (int k = 0; k < 12; k++) w1[k] = P[OW1 + col * NF + 2 * k + half];
#pragma unroll
    for (int r = 0; r < 16; r++) {
        w2[r] = P[OW2 + col * NH + unit(r)];
        if (GRAD) w2t[r] = P[OW2 + unit(r) * NH + col];
        w3[r] = P[OW3 + unit(r)];
        b1[r] = P[OB1 + unit(r)];
        b2[r] = P[OB2 + unit(r)];
    }
    const float b3 = P[OB3];
    v16f gW1 = {}, gW2 = {};
    float gb1 = 0.f, gb2 = 0.f, gw3 = 0.f, gb3 = 0.f, gl = 0.f;
    // unsigned: a step past the largest int stays past nb
    for (unsigned s0 = blockIdx.x * TS; s0 < (unsigned)nb; s0 += gridDim.x * TS) {
        const unsigned s = s0 + col;
        const bool in = s < (unsigned)nb;
        const long long row = in ? (idx ? idx[s] : s) : 0;
        float x[12];
#pragma unroll
        for (int k = 0; k < 12; k++) x[k] = in ? X[row * NF + 2 * k + half] : 0.f;
        v16f z1 = b1, z2 = b2;
#pragma unroll
        for (int k = 0; k < 12; k++) z1 = __builtin_amdgcn_mfma_f32_32x32x2f32(w1[k], x[k], z1, 0, 0, 0);
        float a1[16], d1[16], a2[16], d2[16];
#pragma unroll
        for (int r = 0; r < 16; r++) gelu_both(z1[r], a1[r], d1[r]);
#pragma unroll
        for (int r = 0; r < 16; r++) z2 = __builtin_amdgcn_mfma_f32_32x32x2f32(w2[r], a1[r], z2, 0, 0, 0);
        float z3 = 0.f;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            gelu_both(z2[r], a2[r], d2[r]);
            z3 += w3[r] * a2[r];
        }
        z3 += __shfl_xor(z3, 32);
        z3 += b3;
        const float pr = 1.f / (1.f + expf(-z3));
        if (!GRAD) {
            if (in && half == 0) prob[s] = pr;
            continue;
        }
        const float yy = in ? y[row] : 0.f;
        const float w = !in ? 0.f : yy > 0.5f ? wpos : 1.f;
        const float eps = 1e-7f;
        const float dz3 = in ? w * (pr - yy) : 0.f;
        if (half == 0) {
            gb3 += dz3;
            if (in) gl += -w * (yy * logf(pr + eps) + (1.f - yy) * logf(1.f - pr + eps));
        }
        v16f da = {};
#pragma unroll
        for (int r = 0; r < 16; r++) {
            d2[r] *= dz3 * w3[r];  // dz2
            da = __builtin_amdgcn_mfma_f32_32x32x2f32(w2t[r], d2[r], da, 0, 0, 0);
        }
        __syncthreads();  // the previous tile's reads are done
#pragma unroll
        for (int k = 0; k < 12; k++) sX[col * TP + 2 * k + half] = x[k];
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int o = col * TP + unit(r);
            // nothing from the lanes past the last sample: their activations (of x =
            // 0) may overflow where the samples' do not, and 0 times that is NaN
            sD1[o] = in ? da[r] * d1[r] : 0.f;  // dz1
            sA1[o] = in ? a1[r] : 0.f;
            sD2[o] = in ? d2[r] : 0.f;
            sG3[o] = in ? dz3 * a2[r] : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 16; k++) {
            const int o = (2 * k + half) * TP + col;
            const float v1 = sD1[o], v2 = sD2[o];
            gW1 = __builtin_amdgcn_mfma_f32_32x32x2f32(v1, col < NF ? sX[o] : 0.f, gW1, 0, 0, 0);
            gW2 = __builtin_amdgcn_mfma_f32_32x32x2f32(v2, sA1[o], gW2, 0, 0, 0);
            gb1 += v1;
            gb2 += v2;
            gw3 += sG3[o];
        }
    }
    if (!GRAD) return;
    gb1 += __shfl_xor(gb1, 32);
    gb2 += __shfl_xor(gb2, 32);
    gw3 += __shfl_xor(gw3, 32);
#pragma unroll
    for (int m = 1; m < 32; m <<= 1) {  // held by the lanes of half 0
        gb3 += __shfl_xor(gb3, m);
        gl += __shfl_xor(gl, m);
    }
    float* o = part + (long long)blockIdx.x * PART;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        if (col < NF) o[OW1 + unit(r) * NF + col] = gW1[r];
        o[OW2 + unit(r) * NH + col] = gW2[r];
    }
    if (half == 0) {
        o[OB1 + col] = gb1;
        o[OB2 + col] = gb2;
        o[OW3 + col] = gw3;
    }
    if (lane == 0) {
        o[OB3] = gb3;
        o[MLP_NPARAM] = gl;
    }
}

// Batch-mean gradient (and loss) from nw partial vectors: a block owns 64
// parameters, slice t sums partials t, t + 16, ... in order, the slices are
// added in order; then (adam_t > 0) the Adam update of the parameter.
__global__ void __launch_bounds__(64 * UPD_SLICES) k_mlp_update(float* __restrict__ P, const float* __restrict__ part,
                                                                int nw, int nb, float* __restrict__ grad,
                                                                float* __restrict__ m1, float* __restrict__ m2,
                                                                int adam_t, float lr, float* loss) {
    __shared__ float sum[UPD_SLICES][64];
    const int c = threadIdx.x, t = threadIdx.y, p = blockIdx.x * 64 + c;
    float g = 0.f;
    if (p < PART)
        for (int w = t; w < nw; w += UPD_SLICES) g += part[(long long)w * PART + p];
    sum[t][c] = g;
    __syncthreads();
    if (t != 0 || p >= PART) return;
    for (int q = 1; q < UPD_SLICES; q++) g += sum[q][c];
    const float gr = g * (1.f / (float)nb);
    if (p == MLP_NPARAM) {
        *loss = gr;
        return;
    }
    if (grad) grad[p] = gr;
    if (adam_t > 0) {
        const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
        const float mm = b1 * m1[p] + (1.f - b1) * gr;
        const float vv = b2 * m2[p] + (1.f - b2) * gr * gr;
        m1[p] = mm;
        m2[p] = vv;
        const float mh = mm / (1.f - powf(b1, (float)adam_t));
        const float vh = vv / (1.f - powf(b2, (float)adam_t));
        P[p] -= lr * mh / (sqrtf(vh) + eps);
    }
}

template <typename S>
FeatIn<S> feat_in(const MlpSensorArgsT<S>& a) {
    FeatIn<S> F;
    F.g = a.g;
    F.d = a.d; F.u = a.u; F.v = a.v; F.w = a.w; F.T = a.T;
    for (int m = 0; m < M_COUNT; m++) F.M[m] = a.M[m];
    F.p00 = a.c.p00;
    F.rama = a.c.rama;
    return F;
}

}  // namespace

template <typename S>
void launch_mlp_sensor(const MlpSensorArgsT<S>& a, int plane, hipStream_t st) {
    const Geo& g = a.g;
    dim3 grid;
    if (plane == 0) grid = dim3((g.nx + 1 + 63) / 64, (g.ny + 1 + 3) / 4, g.nz + 1);
    else if (plane == 1) grid = dim3((g.nx + 63) / 64, (g.nz + 3) / 4, 1);
    else grid = dim3((g.nx + 63) / 64, (g.ny + 3) / 4, 1);
    hipLaunchKernelGGL(k_mlp_sensor<S>, grid, dim3(64, 4), 0, st, feat_in(a), a.params, a.c.hy_i1, a.c.hy_i2, a.lo,
                       a.hi, a.fx, a.fy, a.fz, a.prob, plane);
}

template <typename S>
void launch_mlp_collect(const MlpSensorArgsT<S>& a, int stride, float* X, float* y, hipStream_t st) {
    const Geo& g = a.g;
    const int nlx = (g.nx + stride - 1) / stride, nly = (g.ny + stride - 1) / stride, nlz = (g.nz + stride - 1) / stride;
    const long long n = (long long)nlx * nly * nlz;
    hipLaunchKernelGGL(k_mlp_collect<S>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, feat_in(a), stride, nlx,
                       nly, nlz, a.c.hy_i1, a.c.hy_i2, X, y);
}

void launch_mlp_pack(const float* params, float* packed, hipStream_t st) {
    hipLaunchKernelGGL(k_mlp_pack, dim3(1), dim3(64), 0, st, params, packed);
}

long long mlp_collect_count(const Geo& g, int stride) {
    return (long long)((g.nx + stride - 1) / stride) * ((g.ny + stride - 1) / stride) * ((g.nz + stride - 1) / stride);
}

void launch_mlp_step(float* params, const float* X, const float* y, const int* idx, int nb, float wpos, float* part,
                     float* grad, float* m1, float* m2, int adam_t, float lr, float* loss, hipStream_t st) {
    const int nw = mlp_waves(nb);
    hipLaunchKernelGGL(k_mlp_grad<true>, dim3(nw), dim3(64), 0, st, params, X, y, idx, nb, wpos, part, nullptr);
    hipLaunchKernelGGL(k_mlp_update, dim3((PART + 63) / 64), dim3(64, UPD_SLICES), 0, st, params, part, nw, nb, grad,
                       m1, m2, adam_t, lr, loss);
}

void launch_mlp_predict(const float* params, const float* X, int nb, float* prob, hipStream_t st) {
    hipLaunchKernelGGL(k_mlp_grad<false>, dim3(mlp_waves(nb)), dim3(64), 0, st, params, X, nullptr, nullptr, nb, 1.f,
                       nullptr, prob);
}

size_t mlp_part_floats(int nb) { return (size_t)mlp_waves(nb) * PART; }

template void launch_mlp_sensor<double>(const MlpSensorArgsT<double>&, int, hipStream_t);
template void launch_mlp_sensor<float>(const MlpSensorArgsT<float>&, int, hipStream_t);
template void launch_mlp_collect<double>(const MlpSensorArgsT<double>&, int, float*, float*, hipStream_t);
template void launch_mlp_collect<float>(const MlpSensorArgsT<float>&, int, float*, float*, hipStream_t);
