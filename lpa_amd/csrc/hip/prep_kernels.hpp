// prep_kernels.hpp -- one-time graph preparation on the device: record
// validation with degrees and cost features, and the bin-ordered relayout
// of the CGR stream.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cgr_decode.hpp"

namespace lpa {

constexpr int NFEAT = 8;

// Bounds-checked serial reader: every code must end at or before `lim`.
struct SafeReader {
    const uint64_t *W;
    uint64_t pos, lim;
    bool bad;
    __device__ uint64_t window() const {
        uint64_t i = pos >> 6;
        uint32_t s = (uint32_t)(pos & 63);
        return s ? (W[i] << s) | (W[i + 1] >> (64 - s)) : W[i];
    }
    __device__ uint32_t gamma() {
        if (bad || pos >= lim) { bad = true; return 0; }
        uint64_t x = window();
        uint32_t L = (uint32_t)__builtin_clzll(x | 1ull);
        if (L > 31 || pos + 2 * L + 1 > lim) { bad = true; return 0; }
        uint64_t y = x >> (64 - (2 * L + 1));
        pos += 2 * L + 1;
        return (uint32_t)(y - 1);
    }
    __device__ uint32_t zeta() {
        if (bad || pos >= lim) { bad = true; return 0; }
        uint64_t x = window();
        uint32_t h = (uint32_t)__builtin_clzll(x | 1ull);
        if (h > 10 || pos + 4 * (h + 1) > lim) { bad = true; return 0; }
        uint64_t y = (x << (h + 1)) >> (64 - 3 * (h + 1));
        pos += 4 * (h + 1);
        return (uint32_t)(y - 1);
    }
};

// What a lane found in its segments of a record; `end` is the bit after the
// block's last segment in the lane that read it, 0 in the others.
struct ScanPart {
    uint64_t d, end;
    uint32_t n_itv, n_res, itv_len, bad;
    __device__ __forceinline__ void add(const ScanPart &o) {
        d += o.d;
        end += o.end;
        n_itv += o.n_itv;
        n_res += o.n_res;
        itv_len += o.itv_len;
        bad |= o.bad;
    }
};

// Decodes the record at [start, stop) of vertex v with every bound checked
// (codes inside the record, padded segments inside 256 bits, neighbour ids
// < n, record ends exactly at stop), segments dealt out to the `lanes` lanes
// of a group: a segment's place follows from its number, so only the two
// blocks come one after the other.  combine(part) adds up the group's parts
// and gives every lane the total; every lane of the group calls it, twice.
template <class Combine>
__device__ __forceinline__ bool scan_record(const uint64_t *__restrict__ W, uint64_t start, uint64_t stop, uint32_t v,
                                            uint32_t n, uint32_t lane, uint32_t lanes, Combine &&combine, ScanPart &sum,
                                            uint4 &meta) {
    bool ok = start <= stop && v < n;
    uint64_t block_end = start, rbase = 0;
    meta = make_uint4(0, 0, 0, 0);
    sum = ScanPart{};
    for (int blk = 0; blk < 2; blk++) {
        ScanPart part{};
        if (ok) {
            SafeReader r{W, block_end, stop, false};
            const uint32_t ns = r.gamma() + 1;
            const uint64_t base = r.pos;
            if (r.bad || base + (uint64_t)SEG_BITS * (ns - 1) >= stop + (ns > 1 ? 0 : 1)) {
                part.bad = 1;
            } else {
                if (blk == 0) {
                    meta.x = (uint32_t)(base - start);
                    meta.y = ns;
                } else {
                    rbase = base - start;
                    meta.z = (uint32_t)rbase;
                    meta.w = ns;
                }
            }
            for (uint32_t j = lane; j < ns && !part.bad; j += lanes) {
                r.pos = base + (uint64_t)SEG_BITS * j;
                r.lim = j + 1 < ns ? r.pos + SEG_BITS : stop;
                const uint32_t c = r.gamma();
                if (c > r.lim - r.pos) r.bad = true;
                uint64_t prev = 0;   // blk 0: end of the previous interval; blk 1: the previous id
                for (uint32_t t = 0; t < c && !r.bad; t++) {
                    const uint32_t x = blk == 0 ? r.gamma() : r.zeta();
                    const uint64_t first = (x & 1) ? (uint64_t)v - (x >> 1) - 1 : (uint64_t)v + (x >> 1);
                    if (t == 0 && (x & 1) && (uint64_t)(x >> 1) + 1 > v) r.bad = true;
                    const uint64_t id = t == 0 ? first : prev + x + 1;
                    if (blk == 0) {
                        const uint64_t len = (uint64_t)r.gamma() + MIN_ITV;
                        if (id + len > n) r.bad = true;
                        prev = id + len;
                        part.d += len;
                        part.n_itv++;
                        part.itv_len += (uint32_t)len;
                    } else {
                        if (id >= n) r.bad = true;
                        prev = id;
                        part.d++;
                        part.n_res++;
                    }
                }
                if (r.bad) part.bad = 1;
                if (j == ns - 1) part.end = r.pos;
            }
        }
        part = combine(part);
        block_end = part.end;
        ok = ok && !part.bad;
        part.end = 0;
        sum.add(part);
    }
    // segment metadata holds 32-bit relative offsets
    return ok && block_end == stop && rbase < (1ull << 32);
}

// Validates every record and writes its degree, cost features and segment
// metadata -- {bits from the record start to the first interval segment,
// #interval segments, bits to the first residual segment, #residual
// segments}, which lets a group seek every segment at once; sets *err to 1 +
// position on the first malformed record it sees (any one of them).
// SCAN_G lanes per record; a workgroup then takes its records of more than
// SCAN_LONG bits together, all lanes on one record, so that a hub is not
// left to a few lanes (a lane per record took 8.6 ms on R-MAT 19 and 25 ms on
// a copying graph of 300,000 vertices, the time of their longest records;
// R-MAT 19 now takes 0.27 ms).
constexpr uint32_t SCAN_G = 16;
constexpr uint64_t SCAN_LONG = 64 * SEG_BITS;
__global__ void __launch_bounds__(256) k_scan_records(const uint64_t *__restrict__ W,
                                                      const uint64_t *__restrict__ offs,
                                                      const uint32_t *__restrict__ vid, uint64_t start,
                                                      uint64_t n_c, uint32_t n, uint32_t *__restrict__ deg,
                                                      float *__restrict__ feat, uint4 *__restrict__ meta,
                                                      unsigned long long *__restrict__ err) {
    constexpr uint32_t PER = 256 / SCAN_G;
    __shared__ ScanPart parts[4];
    const uint64_t first = start + (uint64_t)blockIdx.x * PER;
    auto finish = [&](uint64_t p, bool ok, const ScanPart &s, const uint4 &m, uint64_t bits) {
        if (!ok) atomicCAS(err, 0ull, (unsigned long long)p + 1);
        const uint64_t d = ok ? s.d : 0;
        deg[p] = (uint32_t)d;
        meta[p] = m;
        if (feat) {
            float *f = feat + p * NFEAT;
            f[0] = (float)d;
            f[1] = (float)s.n_itv;
            f[2] = (float)s.n_res;
            f[3] = (float)bits;
            f[4] = (float)m.y;
            f[5] = (float)m.w;
            f[6] = s.n_itv ? (float)s.itv_len / (float)s.n_itv : 0.0f;
            f[7] = __log2f(1.0f + (float)d);
        }
    };
    auto wave_sum = [](ScanPart x, int width) {
        for (int o = width / 2; o > 0; o >>= 1) {
            ScanPart y;
            y.d = __shfl_xor(x.d, o, 64);
            y.end = __shfl_xor(x.end, o, 64);
            y.n_itv = __shfl_xor(x.n_itv, o, 64);
            y.n_res = __shfl_xor(x.n_res, o, 64);
            y.itv_len = __shfl_xor(x.itv_len, o, 64);
            y.bad = __shfl_xor(x.bad, o, 64);
            x.add(y);
        }
        return x;
    };
    {
        const uint32_t gl = threadIdx.x % SCAN_G;
        const uint64_t p = first + threadIdx.x / SCAN_G;
        const uint64_t start = p < n_c ? offs[p] : 0, stop = p < n_c ? offs[p + 1] : 0;
        const bool mine = p < n_c && !(start <= stop && stop - start > SCAN_LONG);
        ScanPart s;
        uint4 m;
        // groups without a record of their own pass an empty one
        const bool ok = scan_record(W, mine ? start : 1, mine ? stop : 0, mine ? vid[p] : 0, n, gl, SCAN_G,
                                    [&](const ScanPart &x) { return wave_sum(x, SCAN_G); }, s, m);
        if (mine && gl == 0) finish(p, ok, s, m, stop - start);
    }
    for (uint32_t k = 0; k < PER; k++) {
        const uint64_t p = first + k;
        if (p >= n_c) break;
        const uint64_t start = offs[p], stop = offs[p + 1];
        if (!(start <= stop && stop - start > SCAN_LONG)) continue;   // the same in every lane
        ScanPart s;
        uint4 m;
        const bool ok = scan_record(W, start, stop, vid[p], n, threadIdx.x, 256u,
                                    [&](const ScanPart &x) {
                                        const ScanPart w = wave_sum(x, 64);
                                        __syncthreads();   // the last use of parts[] is over
                                        if ((threadIdx.x & 63) == 0) parts[threadIdx.x >> 6] = w;
                                        __syncthreads();
                                        ScanPart t = parts[0];
                                        for (int i = 1; i < 4; i++) t.add(parts[i]);
                                        return t;
                                    }, s, m);
        if (threadIdx.x == 0) finish(p, ok, s, m, stop - start);
    }
}

// Copies `len` bits from bit `s` of src to bit `t` of dst (dst zeroed
// beforehand; words shared with neighbouring records are ORed atomically).
__device__ void copy_bits(const uint64_t *__restrict__ src, uint64_t s, uint64_t *dst, uint64_t t, uint64_t len) {
    for (uint64_t i = 0; i < len; i += 64) {
        const uint32_t c = (uint32_t)(len - i < 64 ? len - i : 64);
        const uint64_t a = s + i;
        const uint32_t sh = (uint32_t)(a & 63);
        uint64_t x = sh ? (src[a >> 6] << sh) | (src[(a >> 6) + 1] >> (64 - sh)) : src[a >> 6];
        if (c < 64) x &= ~0ull << (64 - c);
        const uint64_t b = t + i;
        const uint32_t o = (uint32_t)(b & 63);
        atomicOr((unsigned long long *)&dst[b >> 6], (unsigned long long)(x >> o));
        if (o + c > 64) atomicOr((unsigned long long *)&dst[(b >> 6) + 1], (unsigned long long)(x << (64 - o)));
    }
}

// new position q takes old position perm[q]: record bits, offset, vertex id.
__global__ void __launch_bounds__(256) k_relayout(const uint64_t *__restrict__ W, const uint64_t *__restrict__ offs,
                                                  const uint32_t *__restrict__ vid, const uint4 *__restrict__ meta,
                                                  const uint32_t *__restrict__ perm,
                                                  const uint64_t *__restrict__ new_offs, uint64_t *new_W,
                                                  uint32_t *__restrict__ new_vid, uint4 *__restrict__ new_meta,
                                                  uint64_t n_c) {
    const uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n_c) return;
    const uint32_t p = perm[q];
    new_vid[q] = vid[p];
    new_meta[q] = meta[p];
    copy_bits(W, offs[p], new_W, new_offs[q], offs[p + 1] - offs[p]);
}

// Big-endian 32-bit words (File::graph) -> 64-bit words of the same bit order.
__global__ void k_pack64(const uint32_t *__restrict__ w32, uint64_t n32, uint64_t *__restrict__ w64, uint64_t n64) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n64) return;
    uint64_t hi = 2 * i < n32 ? w32[2 * i] : 0, lo = 2 * i + 1 < n32 ? w32[2 * i + 1] : 0;
    w64[i] = (hi << 32) | lo;
}

__global__ void k_gather_u4(const uint4 *__restrict__ src, const uint32_t *__restrict__ idx, uint32_t n,
                            uint4 *__restrict__ out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = src[idx[i]];
}

// plain copy, 16 bytes per lane (counter calibration)
__global__ void __launch_bounds__(256) k_calibration_copy(const uint4 *__restrict__ src, uint4 *__restrict__ dst,
                                                          uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

// random row gathers (measurement): lane i reads `per_lane` rows of
// W 32-bit words at uniformly random row indices of a buffer of nrows rows
// (indices from a counter-based splitmix64 stream, so no load depends on
// another) and stores one folded word, so the loads cannot be dropped; the
// pattern of the label-row gathers of a step, at a rate the kernels can be
// compared with
template <int W>
__global__ void __launch_bounds__(256) k_calibration_gather(const uint32_t *__restrict__ src, uint64_t nrows,
                                                            uint32_t per_lane, uint64_t seed,
                                                            uint32_t *__restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t acc = 0;
#pragma unroll 8
    for (uint32_t k = 0; k < per_lane; k++) {
        uint64_t z = seed + (i * per_lane + k + 1) * 0x9E3779B97F4A7C15ull;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        const uint32_t *row = src + (z % nrows) * W;
        if (W % 4 == 0) {
#pragma unroll
            for (int q = 0; q < W / 4; q++) {
                const uint4 w = reinterpret_cast<const uint4 *>(row)[q];
                acc ^= w.x ^ w.y ^ w.z ^ w.w;
            }
        } else {
#pragma unroll
            for (int q = 0; q < W; q++) acc ^= row[q];
        }
    }
    out[i] = acc;
}

// Start labels into both label buffers (n*K words each): word i gets vertex
// i / K, or'ed with `seed` (the clamp bit in semi-supervised mode).  Bound by
// the stores: 134 MB per buffer (4 M vertices, 8 vectors) in 0.06 ms, where
// filling on the host, uploading twice and allocating anew took 48 ms.
__global__ void __launch_bounds__(256) k_labels_own(uint32_t *__restrict__ a, uint32_t *__restrict__ b,
                                                    uint64_t first, uint64_t tot, uint32_t K, uint32_t seed) {
    const uint64_t i0 = first + 4 * ((uint64_t)blockIdx.x * 256 + threadIdx.x);
    if (i0 >= tot) return;
    uint32_t v = (uint32_t)(i0 / K), k = (uint32_t)(i0 - (uint64_t)v * K), x[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        x[j] = v | seed;
        if (++k == K) {
            k = 0;
            v++;
        }
    }
    if (i0 + 4 <= tot) {
        *reinterpret_cast<uint4 *>(a + i0) = make_uint4(x[0], x[1], x[2], x[3]);
        *reinterpret_cast<uint4 *>(b + i0) = make_uint4(x[0], x[1], x[2], x[3]);
    } else {
        for (int j = 0; i0 + j < tot; j++) a[i0 + j] = b[i0 + j] = x[j];
    }
}

// Given start labels (already in a): labelled entries of a get `seed` or'ed
// in, and b becomes a copy.
__global__ void __launch_bounds__(256) k_labels_given(uint32_t *__restrict__ a, uint32_t *__restrict__ b,
                                                      uint64_t first, uint64_t tot, uint32_t seed) {
    const uint64_t i0 = first + 4 * ((uint64_t)blockIdx.x * 256 + threadIdx.x);
    if (i0 >= tot) return;
    auto mark = [&](uint32_t x) { return x == 0xFFFFFFFFu ? x : x | seed; };
    if (i0 + 4 <= tot) {
        uint4 x = *reinterpret_cast<uint4 *>(a + i0);
        x = make_uint4(mark(x.x), mark(x.y), mark(x.z), mark(x.w));
        if (seed) *reinterpret_cast<uint4 *>(a + i0) = x;
        *reinterpret_cast<uint4 *>(b + i0) = x;
    } else {
        for (uint64_t i = i0; i < tot; i++) a[i] = b[i] = mark(a[i]);
    }
}

// End of a step's work on a stream: change count l (slots at count + l *
// slots * stride), one per workgroup of 64 lanes, is added up for the host's
// (pinned) word and starts again at 0, in place of a clear before the step and
// a copy after it.
__global__ void __launch_bounds__(64) k_publish(unsigned long long *count, uint32_t slots, uint32_t stride,
                                                unsigned long long *host) {
    unsigned long long *c = count + (uint64_t)blockIdx.x * slots * stride, x = 0;
    for (uint32_t i = threadIdx.x; i < slots; i += 64) {
        x += c[i * stride];
        c[i * stride] = 0;
    }
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    if (threadIdx.x == 0) host[blockIdx.x] = x;
}

__global__ void k_fill_u64(unsigned long long *p, uint64_t n, unsigned long long v) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

}  // namespace lpa
