// mlp_kernels.hpp -- the learned cost model: an 8 -> 32 -> 32 -> 3 MLP
// (ReLU hidden layers, linear outputs) that predicts, for one vertex, the
// log2 of the lane-cycles each of three kernel families would spend on it
// (0: the wave-level kernels, 1: the workgroup kernel with an LDS table,
// 2: the chunked heavy-vertex kernels).  It has no reference counterpart:
// the reference bins by fixed degree thresholds (utils.h:44-85,
// nova_propogator.cuh:210-311).
//
// Kernels (FP32):
//   k_mlp_forward   y = f(x) for n samples, one lane per sample
//   k_mlp_step      one training batch: the Adam update of the previous batch,
//                   then the mean-squared error over the measured outputs
//                   (mask) and its gradient, on the matrix cores
//   k_mlp_sum       loss and gradient of a batch from the workgroups' partials
// Parameter layout (floats): W1[32][8] b1[32] W2[32][32] b2[32] W3[3][32] b3[3].
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lpa {

constexpr int MLP_IN = 8, MLP_H = 32, MLP_OUT = 3;
constexpr int MLP_W1 = 0, MLP_B1 = MLP_W1 + MLP_H * MLP_IN, MLP_W2 = MLP_B1 + MLP_H,
              MLP_B2 = MLP_W2 + MLP_H * MLP_H, MLP_W3 = MLP_B2 + MLP_H, MLP_B3 = MLP_W3 + MLP_OUT * MLP_H,
              MLP_NPARAM = MLP_B3 + MLP_OUT;

struct MlpAct {
    float h1[MLP_H], h2[MLP_H], y[MLP_OUT];
};

__device__ __forceinline__ void mlp_eval(const float *__restrict__ P, const float *x, MlpAct &a) {
#pragma unroll
    for (int j = 0; j < MLP_H; j++) {
        float s = P[MLP_B1 + j];
#pragma unroll
        for (int i = 0; i < MLP_IN; i++) s += P[MLP_W1 + j * MLP_IN + i] * x[i];
        a.h1[j] = s > 0.f ? s : 0.f;
    }
#pragma unroll
    for (int j = 0; j < MLP_H; j++) {
        float s = P[MLP_B2 + j];
#pragma unroll
        for (int i = 0; i < MLP_H; i++) s += P[MLP_W2 + j * MLP_H + i] * a.h1[i];
        a.h2[j] = s > 0.f ? s : 0.f;
    }
#pragma unroll
    for (int j = 0; j < MLP_OUT; j++) {
        float s = P[MLP_B3 + j];
#pragma unroll
        for (int i = 0; i < MLP_H; i++) s += P[MLP_W3 + j * MLP_H + i] * a.h2[i];
        a.y[j] = s;
    }
}

__global__ void __launch_bounds__(256) k_mlp_forward(const float *__restrict__ params, const float *__restrict__ x,
                                                     float *__restrict__ y, uint64_t n) {
    __shared__ float P[MLP_NPARAM];
    for (int i = threadIdx.x; i < MLP_NPARAM; i += blockDim.x) P[i] = params[i];
    __syncthreads();
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    float xi[MLP_IN];
#pragma unroll
    for (int i = 0; i < MLP_IN; i++) xi[i] = x[t * MLP_IN + i];
    MlpAct a;
    mlp_eval(P, xi, a);
#pragma unroll
    for (int j = 0; j < MLP_OUT; j++) y[t * MLP_OUT + j] = a.y[j];
}

using f32x4 = __attribute__((__vector_size__(4 * sizeof(float)))) float;

// Floats of a state array (parameters, first or second moments) and of a
// workgroup's partial: MLP_NPARAM values and, in a partial, the loss after
// them (a multiple of 4 for 16-byte accesses).
constexpr int MLP_STRIDE = 1444;
static_assert(MLP_NPARAM + 1 == MLP_STRIDE && MLP_STRIDE % 4 == 0, "the loss follows the gradient");
constexpr int MLP_WAVES = 4;                  // waves of a k_mlp_step workgroup
constexpr int MLP_TILE = 16;                  // samples per wave and round (one MFMA tile)

// Adam of one step; c1 = 1/(1-b1^t), c2 = 1/(1-b2^t) are its bias corrections.
struct AdamArgs {
    float lr, b1, b2, eps, c1, c2;
};
__device__ __forceinline__ void adam_update(const AdamArgs &k, float g, float &p, float &m1, float &m2) {
    const float a = k.b1 * m1 + (1.f - k.b1) * g;
    const float b = k.b2 * m2 + (1.f - k.b2) * g * g;
    m1 = a;
    m2 = b;
    const float ah = a * k.c1;
    const float bh = b * k.c2;
    p -= k.lr * ah / (sqrtf(bh) + k.eps);
}

// Sum over the partials of the four values at 4 * i4, in a fixed order
// (four interleaved sums, so that the loads do not wait for each other).
__device__ __forceinline__ f32x4 mlp_sum_partials(const float *__restrict__ part, uint32_t np, int i4) {
    f32x4 s[4] = {};
    const f32x4 *src = reinterpret_cast<const f32x4 *>(part) + i4;
    uint32_t w = 0;
    for (; w + 8 <= np; w += 8) {
        f32x4 x[8];
#pragma unroll
        for (int u = 0; u < 8; u++) x[u] = src[(uint64_t)(w + u) * (MLP_STRIDE / 4)];
#pragma unroll
        for (int u = 0; u < 8; u++) s[u & 3] += x[u];
    }
    for (; w < np; w++) s[w & 3] += src[(uint64_t)w * (MLP_STRIDE / 4)];
    return (s[0] + s[1]) + (s[2] + s[3]);
}

// LDS of k_mlp_step: the weights with rows padded against bank conflicts
// (W3 to 16 rows, the last 13 zero), and per wave a staging area of the
// tile's values, one row per feature with its 16 samples (stride 20: rows
// 16-byte aligned, four samples per read).
struct MlpShared {
    static constexpr int S2 = 36, SROW = 20;
    static constexpr int DZ2 = 0, H1 = 32, DZ1 = 64, X = 96, DY = 112, H2 = 128, ROWS = 160;
    float w1[MLP_H * MLP_IN], b1[MLP_H], w2[MLP_H * S2], b2[MLP_H], w3[16 * S2], b3[16];
    __align__(16) float stage[MLP_WAVES][ROWS * SROW];
    __device__ __forceinline__ void put(int i, float p) {
        if (i < MLP_B1) w1[i] = p;
        else if (i < MLP_W2) b1[i - MLP_B1] = p;
        else if (i < MLP_B2) w2[((i - MLP_W2) / MLP_H) * S2 + (i - MLP_W2) % MLP_H] = p;
        else if (i < MLP_W3) b2[i - MLP_B2] = p;
        else if (i < MLP_B3) w3[((i - MLP_W3) / MLP_H) * S2 + (i - MLP_W3) % MLP_H] = p;
        else b3[i - MLP_B3] = p;
    }
};
static_assert(MLP_WAVES * MLP_STRIDE <= MLP_WAVES * MlpShared::ROWS * MlpShared::SROW, "partials reuse the staging area");

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// One training batch.  First every workgroup sums the previous batch's
// partials (np of them; 0: no update pending) and applies Adam to all 1,443
// parameters for itself (workgroup 0 also stores the new state in `next` and
// adds the batch's loss to *loss): a redundant update costs less than a
// launch or a grid barrier between batches.  Then loss = sum over samples and
// masked outputs of (y - target)^2 * scale and its gradient over samples
// idx[0..n) (or 0..n-1), of which every workgroup leaves its share in
// part_out.
//
// A wave takes 16 samples at a time, and every product runs on the matrix
// cores in FP32 (16x16x4 tiles): activations are held as [feature][sample]
// tiles, whose accumulator registers (rows 4g + r of lane group g) are used
// as the next product's operand as they are, with the weights read in the
// same order of the inner index.  Only the gradients, which contract over
// the samples, need the transposed tiles: they pass through LDS.  Biases
// take a constant-one feature (row 8 of the inputs' tile).
//
// Bound by latency: a batch of 2048 samples is 32 workgroups of 4 waves.
// Training on 200,000 samples, two epochs at batch 2048: 3.4 ms, against 255
// ms with a lane per sample adding its 1,443 products to LDS with atomics
// (1.6 ms per batch: every lane of a wave on the same address).
__global__ void __launch_bounds__(64 * MLP_WAVES) k_mlp_step(
    const float *__restrict__ cur, float *__restrict__ next, const float *__restrict__ part_in, uint32_t np,
    AdamArgs adam, double *__restrict__ loss, const float *__restrict__ x, const float *__restrict__ target,
    const uint8_t *__restrict__ mask, const uint32_t *__restrict__ idx, uint64_t n, float scale,
    float *__restrict__ part_out) {
    __shared__ MlpShared sh;
    using M = MlpShared;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
    for (int i = threadIdx.x; i < 13 * M::S2; i += blockDim.x) sh.w3[MLP_OUT * M::S2 + i] = 0.f;
    if (threadIdx.x >= MLP_OUT && threadIdx.x < 16) sh.b3[threadIdx.x] = 0.f;
    float *S = sh.stage[wave];
    // rows that no tile writes: the unused input features and outputs
    for (int i = lane; i < 7 * M::SROW; i += 64) S[(M::X + 9) * M::SROW + i] = 0.f;
    for (int i = lane; i < 13 * M::SROW; i += 64) S[(M::DY + MLP_OUT) * M::SROW + i] = 0.f;
    for (int i4 = threadIdx.x; i4 < MLP_STRIDE / 4; i4 += blockDim.x) {
        f32x4 p = reinterpret_cast<const f32x4 *>(cur)[i4];
        if (np) {
            f32x4 m1 = reinterpret_cast<const f32x4 *>(cur + MLP_STRIDE)[i4];
            f32x4 m2 = reinterpret_cast<const f32x4 *>(cur + 2 * MLP_STRIDE)[i4];
            const f32x4 gr = mlp_sum_partials(part_in, np, i4);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (4 * i4 + j < MLP_NPARAM) {
                    float pj = p[j], aj = m1[j], bj = m2[j];
                    adam_update(adam, gr[j], pj, aj, bj);
                    p[j] = pj;
                    m1[j] = aj;
                    m2[j] = bj;
                } else if (blockIdx.x == 0) {
                    *loss += (double)gr[j];
                }
            }
            if (blockIdx.x == 0) {
                reinterpret_cast<f32x4 *>(next)[i4] = p;
                reinterpret_cast<f32x4 *>(next + MLP_STRIDE)[i4] = m1;
                reinterpret_cast<f32x4 *>(next + 2 * MLP_STRIDE)[i4] = m2;
            }
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (4 * i4 + j < MLP_NPARAM) sh.put(4 * i4 + j, p[j]);
    }
    if (n == 0) return;   // the last update of a run
    __syncthreads();

    f32x4 gw2[2][2] = {}, gw1[2] = {}, gw3[2] = {}, gb2[2] = {}, gb3 = {};
    float lsum = 0.f;
    const uint64_t ntiles = (n + MLP_TILE - 1) / MLP_TILE;
    for (uint64_t tile = (uint64_t)blockIdx.x * MLP_WAVES + wave; tile < ntiles; tile += (uint64_t)gridDim.x * MLP_WAVES) {
        const uint64_t q = tile * MLP_TILE + c;
        const bool valid = q < n;
        const uint64_t t = valid ? (idx ? (uint64_t)idx[q] : q) : 0;
        float x0 = 0.f, x1 = 0.f, tg[MLP_OUT] = {};
        bool mk[MLP_OUT] = {};
        if (valid) {
            x0 = x[t * MLP_IN + 2 * g];
            x1 = x[t * MLP_IN + 2 * g + 1];
            if (g == 0) {
#pragma unroll
                for (int j = 0; j < MLP_OUT; j++) {
                    tg[j] = target[t * MLP_OUT + j];
                    mk[j] = mask[t * MLP_OUT + j] != 0;
                }
            }
        }
        // forward: lane (g, c) holds rows 16 u + 4 g + r of sample c
        float h1[2][4], h2[2][4];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            f32x4 z;
#pragma unroll
            for (int r = 0; r < 4; r++) z[r] = sh.b1[16 * u + 4 * g + r];
            z = mfma4(sh.w1[(16 * u + c) * MLP_IN + 2 * g], x0, z);
            z = mfma4(sh.w1[(16 * u + c) * MLP_IN + 2 * g + 1], x1, z);
#pragma unroll
            for (int r = 0; r < 4; r++) h1[u][r] = z[r] > 0.f ? z[r] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            f32x4 z;
#pragma unroll
            for (int r = 0; r < 4; r++) z[r] = sh.b2[16 * u + 4 * g + r];
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (int r = 0; r < 4; r++) z = mfma4(sh.w2[(16 * u + c) * M::S2 + 16 * k + 4 * g + r], h1[k][r], z);
#pragma unroll
            for (int r = 0; r < 4; r++) h2[u][r] = z[r] > 0.f ? z[r] : 0.f;
        }
        f32x4 y;
#pragma unroll
        for (int r = 0; r < 4; r++) y[r] = sh.b3[4 * g + r];
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
            for (int r = 0; r < 4; r++) y = mfma4(sh.w3[c * M::S2 + 16 * k + 4 * g + r], h2[k][r], y);
        // errors: outputs 0..2 of sample c are in lane group 0
        float dy[MLP_OUT], l = 0.f;
        bool any = false;
#pragma unroll
        for (int j = 0; j < MLP_OUT; j++) {
            const float e = mk[j] ? y[j] - tg[j] : 0.f;
            l += e * e;
            dy[j] = 2.f * e * scale;
            any = any || dy[j] != 0.f;
        }
        lsum += l * scale;
        // a sample without an error contributes nothing, whatever its inputs
        const bool live = __shfl((int)any, c, 64) != 0;
        const float e0 = __shfl(dy[0], c, 64), e1 = __shfl(dy[1], c, 64), e2 = __shfl(dy[2], c, 64);
        const float dyg = g == 0 ? e0 : g == 1 ? e1 : g == 2 ? e2 : 0.f;
        // back through the layers
        float dz2[2][4], dz1[2][4];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const f32x4 z = mfma4(sh.w3[g * M::S2 + 16 * u + c], dyg, f32x4{});
#pragma unroll
            for (int r = 0; r < 4; r++) dz2[u][r] = h2[u][r] > 0.f ? z[r] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            f32x4 z = {};
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (int r = 0; r < 4; r++) z = mfma4(sh.w2[(16 * k + 4 * g + r) * M::S2 + 16 * u + c], dz2[k][r], z);
#pragma unroll
            for (int r = 0; r < 4; r++) dz1[u][r] = h1[u][r] > 0.f ? z[r] : 0.f;
        }
        // stage [feature][sample]
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int f = (16 * u + 4 * g + r) * M::SROW + c;
                S[M::DZ2 * M::SROW + f] = live ? dz2[u][r] : 0.f;
                S[M::DZ1 * M::SROW + f] = live ? dz1[u][r] : 0.f;
                S[M::H1 * M::SROW + f] = live ? h1[u][r] : 0.f;
                S[M::H2 * M::SROW + f] = live ? h2[u][r] : 0.f;
            }
        S[(M::X + 2 * g) * M::SROW + c] = live ? x0 : 0.f;
        S[(M::X + 2 * g + 1) * M::SROW + c] = live ? x1 : 0.f;
        if (g == 0) {
            S[(M::X + 8) * M::SROW + c] = live ? 1.f : 0.f;
#pragma unroll
            for (int j = 0; j < MLP_OUT; j++) S[(M::DY + j) * M::SROW + c] = dy[j];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // gradients: products over the 16 samples, four per lane group
        auto rows = [&](int base) { return *reinterpret_cast<const f32x4 *>(&S[(base + c) * M::SROW + 4 * g]); };
        const f32x4 vx = rows(M::X), vy = rows(M::DY);
        f32x4 a2[2], a1[2], v1[2], v2[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            a2[u] = rows(M::DZ2 + 16 * u);
            a1[u] = rows(M::DZ1 + 16 * u);
            v1[u] = rows(M::H1 + 16 * u);
            v2[u] = rows(M::H2 + 16 * u);
        }
#pragma unroll
        for (int s = 0; s < 4; s++) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
#pragma unroll
                for (int k = 0; k < 2; k++) gw2[u][k] = mfma4(a2[u][s], v1[k][s], gw2[u][k]);
                gw1[u] = mfma4(a1[u][s], vx[s], gw1[u]);
                gb2[u] = mfma4(a2[u][s], vx[s], gb2[u]);
                gw3[u] = mfma4(vy[s], v2[u][s], gw3[u]);
            }
            gb3 = mfma4(vy[s], vx[s], gb3);
        }
        __builtin_amdgcn_wave_barrier();   // the staging rows are written again next round
    }
    // the waves' sums, then the workgroup's partial
    __syncthreads();
    float *R = &sh.stage[0][0] + wave * MLP_STRIDE;
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int f = 16 * u + 4 * g + r;
#pragma unroll
            for (int k = 0; k < 2; k++) R[MLP_W2 + f * MLP_H + 16 * k + c] = gw2[u][k][r];
            if (c < MLP_IN) R[MLP_W1 + f * MLP_IN + c] = gw1[u][r];
            if (c == 8) {
                R[MLP_B1 + f] = gw1[u][r];
                R[MLP_B2 + f] = gb2[u][r];
            }
            if (g == 0 && r < MLP_OUT) R[MLP_W3 + r * MLP_H + 16 * u + c] = gw3[u][r];
        }
    if (g == 0 && c == 8) {
#pragma unroll
        for (int r = 0; r < MLP_OUT; r++) R[MLP_B3 + r] = gb3[r];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o, 64);
    if (lane == 0) R[MLP_NPARAM] = lsum;
    __syncthreads();
    const f32x4 *all = reinterpret_cast<const f32x4 *>(&sh.stage[0][0]);
    for (int i4 = threadIdx.x; i4 < MLP_STRIDE / 4; i4 += blockDim.x) {
        f32x4 s = all[i4];
#pragma unroll
        for (int w = 1; w < MLP_WAVES; w++) s += all[w * (MLP_STRIDE / 4) + i4];
        reinterpret_cast<f32x4 *>(part_out)[(uint64_t)blockIdx.x * (MLP_STRIDE / 4) + i4] = s;
    }
}

// Gradient and loss (MLP_STRIDE floats) of a batch from its partials.
__global__ void __launch_bounds__(64) k_mlp_sum(const float *__restrict__ part, uint32_t np, float *__restrict__ out) {
    const int i4 = blockIdx.x * blockDim.x + threadIdx.x;
    if (i4 < MLP_STRIDE / 4) reinterpret_cast<f32x4 *>(out)[i4] = mlp_sum_partials(part, np, i4);
}

}  // namespace lpa
