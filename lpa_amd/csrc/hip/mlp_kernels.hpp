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
//                   (mask) and its gradient, the layers on the matrix cores
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
constexpr int MLP_CHUNK = MLP_WAVES * MLP_TILE;   // samples per workgroup and round
static_assert(64 * MLP_WAVES == MLP_H * MLP_IN && 64 * MLP_WAVES == 16 * 16, "a lane's sums");

// Adam of one step; c1 = 1/(1-b1^t), c2 = 1/(1-b2^t) are its bias corrections.
// (Which products are fused is spelled out, so that the same bits come from
// every place that this is inlined in.)
struct AdamArgs {
    float lr, b1, b2, eps, c1, c2;
};
__device__ __forceinline__ void adam_update(const AdamArgs &k, float g, float &p, float &m1, float &m2) {
#pragma clang fp contract(off)
    const float a = __builtin_fmaf(1.f - k.b1, g, k.b1 * m1);
    const float b = __builtin_fmaf(g, (1.f - k.b2) * g, k.b2 * m2);
    m1 = a;
    m2 = b;
    const float ah = a * k.c1;
    const float bh = b * k.c2;
    p -= k.lr * ah / (sqrtf(bh) + k.eps);
}

// Sum over the partials of the four values at 4 * i4: four partials (256
// samples) together, then those sums one after the other.
__device__ __forceinline__ f32x4 mlp_sum_partials(const float *__restrict__ part, uint32_t np, int i4) {
    f32x4 s = {};
    const f32x4 *src = reinterpret_cast<const f32x4 *>(part) + i4;
    uint32_t w = 0;
    for (; w + 8 <= np; w += 8) {
        f32x4 x[8];
#pragma unroll
        for (int u = 0; u < 8; u++) x[u] = src[(uint64_t)(w + u) * (MLP_STRIDE / 4)];
        s += ((x[0] + x[1]) + x[2]) + x[3];
        s += ((x[4] + x[5]) + x[6]) + x[7];
    }
    while (w < np) {
        f32x4 x = src[(uint64_t)w++ * (MLP_STRIDE / 4)];
        for (; w < np && w % 4; w++) x += src[(uint64_t)w * (MLP_STRIDE / 4)];
        s += x;
    }
    return s;
}

// LDS of k_mlp_step: the weights with rows padded against bank conflicts
// (W3 to 16 rows, the last 13 zero), and per wave a staging area of its 16
// samples' values, one row per feature (stride 20: rows 16-byte aligned, four
// samples per read, and 16 rows side by side meet every bank once).
struct MlpShared {
    static constexpr int S2 = 36, SROW = 20;
    static constexpr int DZ2 = 0, H1 = 32, DZ1 = 64, H2 = 96, X = 128, ONE = 136, DY = 137, ROWS = 140;
    float w1[MLP_H * MLP_IN], b1[MLP_H], w2[MLP_H * S2], b2[MLP_H], w3[16 * S2], b3[16];
    float loss[MLP_WAVES];
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

// Feature in row m of a 16-row accumulator or weight tile (its own inverse).
__device__ __forceinline__ int mlp_feature(int m) { return 4 * (m & 3) + (m >> 2); }

// One more term of a gradient, its product rounded first.
__device__ __forceinline__ void mlp_add(float &acc, float a, float b) {
#pragma clang fp contract(off)
    const float p = a * b;
    acc += p;
}

__device__ __forceinline__ bool mlp_finite(f32x4 x) {
    return x[0] * 0.f + x[1] * 0.f + x[2] * 0.f + x[3] * 0.f == 0.f;   // an infinity times 0 is NaN
}

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
// A workgroup takes 64 samples at a time, a wave 16 of them, whose way through
// the layers and back runs on the matrix cores in FP32 (16x16x4 tiles):
// activations are held as [feature][sample] tiles, whose accumulator registers
// are used as the next product's operand as they are.
//
// Every sum is taken in the order of a lane that walks over the layers sample
// by sample, bit for bit.  That matters where a pre-activation is a rounding
// away from 0: another order flips the unit, and Adam turns the lone gradient
// of a nearly dead unit into a full step (parameters 5e-5 apart after two
// epochs of 98 batches, 1e-7 otherwise).  An MFMA adds its four products to the
// accumulator one after the other, lane group 0 first, each as a fused
// multiply-add, so features are placed such that every product takes its
// inputs in ascending order: accumulator row 4g + r (register r of lane group
// g) is feature 4r + g (mlp_feature), and register r of the groups is then the
// next four inputs.  The gradients, which contract over the samples, go
// through LDS to the vector units: a rounded product and a sum per sample, in
// the samples' order (5.6 of the 1,443 sums per lane; a contraction on the
// matrix cores fuses them and takes 0.75 us less per batch).  64 samples make a
// partial, four partials are summed before they join the others.
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
    const int f = mlp_feature(c);   // the feature whose weights this lane passes
    for (int i = threadIdx.x; i < 13 * M::S2; i += blockDim.x) sh.w3[MLP_OUT * M::S2 + i] = 0.f;
    if (threadIdx.x >= MLP_OUT && threadIdx.x < 16) sh.b3[threadIdx.x] = 0.f;
    float *S = sh.stage[wave];
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

    // this lane's sums: four weights of the second layer, one of the first,
    // and one of the third or a bias, as products of two staged rows
    const int t4 = threadIdx.x >> 4, t8 = threadIdx.x >> 3;
    int ra = M::X, rb = M::X, out = -1;
    if (threadIdx.x < 96) {
        ra = M::DY + (threadIdx.x >> 5), rb = M::H2 + (threadIdx.x & 31), out = MLP_W3 + threadIdx.x;
    } else if (threadIdx.x < 160) {
        const int j = threadIdx.x & 31;
        ra = (threadIdx.x < 128 ? M::DZ1 : M::DZ2) + j, rb = M::ONE, out = (threadIdx.x < 128 ? MLP_B1 : MLP_B2) + j;
    } else if (threadIdx.x < 160 + MLP_OUT) {
        ra = M::DY + threadIdx.x - 160, rb = M::ONE, out = MLP_B3 + threadIdx.x - 160;
    }
    float total[6] = {}, lsum = 0.f;
    const uint64_t chunks = (n + MLP_CHUNK - 1) / MLP_CHUNK;
    for (uint64_t chunk = blockIdx.x; chunk < chunks; chunk += gridDim.x) {
        const uint64_t q = chunk * MLP_CHUNK + wave * MLP_TILE + c;
        const bool valid = q < n;
        const uint64_t t = valid ? (idx ? (uint64_t)idx[q] : q) : 0;
        float x0 = 0.f, x1 = 0.f, tg[MLP_OUT] = {};
        bool mk[MLP_OUT] = {};
        if (valid) {
            x0 = x[t * MLP_IN + g];
            x1 = x[t * MLP_IN + 4 + g];
            if (g == 0) {
#pragma unroll
                for (int j = 0; j < MLP_OUT; j++) {
                    tg[j] = target[t * MLP_OUT + j];
                    mk[j] = mask[t * MLP_OUT + j] != 0;
                }
            }
        }
        // forward: lane (g, c) holds features 16 u + 4 r + g of sample c
        float h1[2][4], h2[2][4];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            f32x4 z;
#pragma unroll
            for (int r = 0; r < 4; r++) z[r] = sh.b1[16 * u + 4 * r + g];
            z = mfma4(sh.w1[(16 * u + f) * MLP_IN + g], x0, z);
            z = mfma4(sh.w1[(16 * u + f) * MLP_IN + 4 + g], x1, z);
#pragma unroll
            for (int r = 0; r < 4; r++) h1[u][r] = z[r] > 0.f ? z[r] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            f32x4 z;
#pragma unroll
            for (int r = 0; r < 4; r++) z[r] = sh.b2[16 * u + 4 * r + g];
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (int r = 0; r < 4; r++) z = mfma4(sh.w2[(16 * u + f) * M::S2 + 16 * k + 4 * r + g], h1[k][r], z);
#pragma unroll
            for (int r = 0; r < 4; r++) h2[u][r] = z[r] > 0.f ? z[r] : 0.f;
        }
        f32x4 y;
#pragma unroll
        for (int r = 0; r < 4; r++) y[r] = sh.b3[4 * g + r];   // outputs in row order: only three
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
            for (int r = 0; r < 4; r++) y = mfma4(sh.w3[c * M::S2 + 16 * k + 4 * r + g], h2[k][r], y);
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
        f32x4 dz2[2], dz1[2];
#pragma unroll
        for (int u = 0; u < 2; u++) dz2[u] = mfma4(sh.w3[g * M::S2 + 16 * u + f], dyg, f32x4{});
        if (__any(!mlp_finite(dz2[0]) || !mlp_finite(dz2[1]))) {   // rare: 0 times a weight that is not finite counts as 0
#pragma unroll
            for (int u = 0; u < 2; u++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float *w = &sh.w3[16 * u + 4 * r + g];
                    float z = e0 != 0.f ? e0 * w[0] : 0.f;
                    if (e1 != 0.f) z = __builtin_fmaf(e1, w[M::S2], z);
                    if (e2 != 0.f) z = __builtin_fmaf(e2, w[2 * M::S2], z);
                    dz2[u][r] = z;
                }
        }
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) dz2[u][r] = h2[u][r] > 0.f ? dz2[u][r] : 0.f;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            dz1[u] = f32x4{};
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    dz1[u] = mfma4(sh.w2[(16 * k + 4 * r + g) * M::S2 + 16 * u + f], dz2[k][r], dz1[u]);
        }
        if (__any(!mlp_finite(dz1[0]) || !mlp_finite(dz1[1]))) {
#pragma unroll
            for (int u = 0; u < 2; u++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    S[(M::DZ2 + 16 * u + 4 * r + g) * M::SROW + c] = dz2[u][r];
                    dz1[u][r] = 0.f;
                }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll 1
            for (int j = 0; j < MLP_H; j++) {
                const float d = S[(M::DZ2 + j) * M::SROW + c];
                if (d == 0.f) continue;
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int r = 0; r < 4; r++) dz1[u][r] = __builtin_fmaf(sh.w2[j * M::S2 + 16 * u + 4 * r + g], d, dz1[u][r]);
            }
            __builtin_amdgcn_wave_barrier();   // the rows are written again below
        }
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) dz1[u][r] = h1[u][r] > 0.f ? dz1[u][r] : 0.f;
        // stage [feature][sample]
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int at = (16 * u + 4 * r + g) * M::SROW + c;
                S[M::DZ2 * M::SROW + at] = live ? dz2[u][r] : 0.f;
                S[M::DZ1 * M::SROW + at] = live ? dz1[u][r] : 0.f;
                S[M::H1 * M::SROW + at] = live ? h1[u][r] : 0.f;
                S[M::H2 * M::SROW + at] = live ? h2[u][r] : 0.f;
            }
        S[(M::X + g) * M::SROW + c] = live ? x0 : 0.f;
        S[(M::X + 4 + g) * M::SROW + c] = live ? x1 : 0.f;
        if (g == 0) {
            S[M::ONE * M::SROW + c] = live ? 1.f : 0.f;
#pragma unroll
            for (int j = 0; j < MLP_OUT; j++) S[(M::DY + j) * M::SROW + c] = dy[j];
        }
        __syncthreads();
        float acc[6];
        auto sums = [&](auto add) {
#pragma unroll
            for (int i = 0; i < 6; i++) acc[i] = 0.f;
            for (int w = 0; w < MLP_WAVES; w++)
#pragma unroll
                for (int s = 0; s < MLP_TILE; s += 4) {
                    auto row = [&](int i) { return *reinterpret_cast<const f32x4 *>(&sh.stage[w][i * M::SROW + s]); };
                    const f32x4 a0 = row(M::DZ2 + t4), a1 = row(M::DZ2 + 16 + t4), a2 = row(M::DZ1 + t8), a3 = row(ra);
                    const f32x4 v0 = row(M::H1 + c), v1 = row(M::H1 + 16 + c), v2 = row(M::X + (lane & 7)), v3 = row(rb);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        add(acc[0], a0[e], v0[e]);
                        add(acc[1], a0[e], v1[e]);
                        add(acc[2], a1[e], v0[e]);
                        add(acc[3], a1[e], v1[e]);
                        add(acc[4], a2[e], v2[e]);
                        add(acc[5], a3[e], v3[e]);
                    }
                }
        };
        sums([](float &s, float a, float b) { mlp_add(s, a, b); });
        if (!mlp_finite(f32x4{acc[0], acc[1], acc[2], acc[3]}) || !mlp_finite(f32x4{acc[4], acc[5], 0.f, 0.f})) {
            asm volatile("" ::: "memory");          // the rows are read again, not kept in 512 registers
            sums([](float &s, float a, float b) {   // rare, as above: the gradient's factor decides
                if (a != 0.f) mlp_add(s, a, b);
            });
        }
#pragma unroll
        for (int i = 0; i < 6; i++) total[i] += acc[i];
        __syncthreads();   // the staging rows are written again next round
    }
    // the workgroup's partial
    float *R = part_out + (uint64_t)blockIdx.x * MLP_STRIDE;
#pragma unroll
    for (int i = 0; i < 4; i++) R[MLP_W2 + (t4 + 16 * (i >> 1)) * MLP_H + c + 16 * (i & 1)] = total[i];
    R[MLP_W1 + threadIdx.x] = total[4];
    if (out >= 0) R[out] = total[5];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o, 64);
    if (lane == 0) sh.loss[wave] = lsum;
    __syncthreads();
    if (threadIdx.x == 0) R[MLP_NPARAM] = (sh.loss[0] + sh.loss[1]) + (sh.loss[2] + sh.loss[3]);
}

// Gradient and loss (MLP_STRIDE floats) of a batch from its partials.
__global__ void __launch_bounds__(64) k_mlp_sum(const float *__restrict__ part, uint32_t np, float *__restrict__ out) {
    const int i4 = blockIdx.x * blockDim.x + threadIdx.x;
    if (i4 < MLP_STRIDE / 4) reinterpret_cast<f32x4 *>(out)[i4] = mlp_sum_partials(part, np, i4);
}

}  // namespace lpa
