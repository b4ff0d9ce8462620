// encode_wave.hpp -- CGR records encoded by a wave each.
//
// A lane that encodes a record alone walks its row several times, id by id;
// in a power-law graph the lanes with the longest rows keep the kernel busy
// long after the others are done (R-MAT 19: 75 ms for the lengths and 72 ms
// for the bits, against 24 MB of stream).  The kernels here give rows longer
// than LANE_ROW ids to a wave, which reads the row 64 ids at a time, with the
// next 64 already loaded, and keeps everything that the format's rules carry
// from one id to the next in scalar registers:
//
//  - runs: bit i of C says that id i follows id i - 1; three set bits in a
//    row are a run of four, so shifts and ANDs of C with its neighbours'
//    bits give the ids inside runs of >= 4 (interval entries, emitted at the
//    lane where the run ends) and the others (residual entries).
//  - segments: the entries' bits are summed along the wave, and one compare
//    and ballot finds the first entry that overflows the open segment, so a
//    segment costs one round whatever it holds.
//
// Lengths need no memory at all.  To write, the row is streamed again: the
// entries go through a ring in LDS, because a segment starts with its count
// (known when it closes) and the last closed segment takes the open tail as
// well (known at the end of the row); a closed segment is written by the
// whole wave, its codes ORed into an LDS copy of its words.
//
// R-MAT 19 (15.5 M ids, 24 MB of stream), with the workgroup kernels taking
// rows above 8192 ids: lengths 75 -> 0.18 ms and bits 72 -> 0.96 ms here, 0.9
// and 0.05 ms there.  Bound by the latency of the longest wave's rounds (about
// 1.4 us per 64 ids).
#pragma once
#include "encode_kernels.hpp"

namespace lpa {

namespace enc {

// Longest row left to a lane (k_encode_len / k_encode_write); longer ones
// take a wave.  A lane needs several dependent walks over its ids, a wave the
// same time for 1 to 64 ids.
constexpr uint32_t LANE_ROW = 16;
constexpr int ENC_WAVES = 4;          // waves (rows) per workgroup
constexpr uint32_t RING = 512;        // entries; at most 127 + 127 of the last
                                      // closed and the open segment, and 64 new ones
constexpr uint32_t SEG_WORDS = 32;    // 32-bit words of a segment copy (at most
                                      // 2 x 256 bits, a header and the alignment)

__device__ __forceinline__ uint32_t flog2_32(uint32_t y) { return 31u - (uint32_t)__builtin_clz(y); }
__device__ __forceinline__ uint32_t gamma_len32(uint32_t x) { return 2u * flog2_32(x + 1) + 1u; }
__device__ __forceinline__ uint32_t zeta_len32(uint32_t x) { return (flog2_32(x + 1) / 3u + 1u) * 4u; }
__device__ __forceinline__ uint32_t nat32(uint32_t u, uint32_t v) { return u >= v ? (u - v) << 1 : ((v - u) << 1) - 1; }

// inclusive sum over the wave: within rows of 16 lanes, then across them
__device__ __forceinline__ uint32_t wave_scan(uint32_t x) {
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xF, 0xF, false);   // row_shr:1
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xF, 0xF, false);   // row_shr:2
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xF, 0xF, false);   // row_shr:4
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xF, 0xF, false);   // row_shr:8
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xA, 0xF, false);   // row_bcast:15
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xC, 0xF, false);   // row_bcast:31
    return x;
}
__device__ __forceinline__ uint32_t lane_value(uint32_t x, int l) { return (uint32_t)__builtin_amdgcn_readlane((int)x, l); }
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One block's segmentation while its entries stream by (the same in every lane).
struct WaveBlock {
    uint32_t entries = 0, closed = 0;
    uint32_t cnt = 0, cur = 0;                   // open segment: entries, bits
    uint32_t open_idx = 0, open_fb = 0;          // its first entry and that entry's bits
    uint32_t last_idx = 0, last_fb = 0;          // the same of the last closed segment
    uint64_t sum = 0, open_sum = 0, last_sum = 0;   // later-bits of the entries so far; up to those first entries
    // 64 lanes' entries (mask E): bits fb when it opens a segment, and the
    // inclusive sum P of the bits when it follows another.  close(s, e) is
    // called for every segment [s, e) that closes.
    template <class Close>
    __device__ __forceinline__ void feed(uint64_t E, uint32_t P, uint32_t fb, Close &&close) {
        if (E == 0) return;
        const uint32_t lane = __lane_id();
        const uint64_t upto = (2ull << lane) - 1;
        const uint32_t total = lane_value(P, 63);
        uint64_t rem = E;
        uint32_t before = 0;
        if (cnt == 0) {   // the block's first entry
            const int f = __builtin_ctzll(rem);
            open_fb = cur = lane_value(fb, f);
            before = lane_value(P, f);
            open_sum = before;
            cnt = 1;
            rem &= rem - 1;
        }
        while (rem) {
            const bool over = ((rem >> lane) & 1) &&
                              gamma_len32(cnt + (uint32_t)__popcll(rem & upto)) + cur + (P - before) > SEG;
            const uint64_t O = __ballot(over);
            if (O == 0) {
                cnt += (uint32_t)__popcll(rem);
                cur += total - before;
                break;
            }
            const int f = __builtin_ctzll(O);
            const uint32_t idx = entries + (uint32_t)__popcll(E & ((1ull << f) - 1));
            close(open_idx, idx);
            closed++;
            last_idx = open_idx;
            last_fb = open_fb;
            last_sum = open_sum;
            open_idx = idx;
            open_fb = cur = lane_value(fb, f);
            before = lane_value(P, f);
            open_sum = sum + before;
            cnt = 1;
            rem = E & ~((2ull << f) - 1);
        }
        entries += (uint32_t)__popcll(E);
        sum += total;
    }
    __device__ __forceinline__ uint32_t segs() const { return closed ? closed : 1; }
    __device__ __forceinline__ uint32_t tail_idx() const { return closed ? last_idx : 0; }
    __device__ __forceinline__ uint64_t bits() const {
        const uint32_t c = entries - tail_idx();
        uint64_t b = gamma_len32(segs() - 1) + (uint64_t)SEG * (segs() - 1) + gamma_len32(c);
        if (c) b += (closed ? last_fb : open_fb) + (sum - (closed ? last_sum : open_sum));
        return b;
    }
};

// The entries of 64 ids: per lane an interval entry (left, len) where a run
// ends, a residual entry (id) or none; gap = the code when it follows another
// entry of its block (any value for the block's first).
struct WaveChunk {
    uint64_t itv, res;          // lanes with an entry
    uint32_t id, left, len, gap;
};

// Streams row adj[0..d) (strictly increasing) through sink(chunk); with
// CHECK, returns false (and stops) at an id >= n or one that does not
// increase.
template <bool CHECK, class Sink>
__device__ __forceinline__ bool wave_row(const uint32_t *__restrict__ adj, uint32_t d, uint32_t n, Sink &&sink) {
    const uint32_t lane = __lane_id();
    const uint64_t below = (1ull << lane) - 1;
    uint32_t cu = lane < d ? adj[lane] : 0;
    uint32_t prev = 0;                       // last id of the chunk before
    uint64_t C = 0, TP = 0;                  // this chunk's C; four-run starts of the one before
    uint32_t run_left = 0, last_res = 0, last_end = 0;
    {
        const uint32_t pu = (uint32_t)__shfl_up((int)cu, 1, 64);
        C = __ballot(lane < d && lane > 0 && cu == pu + 1);
    }
    for (uint32_t i0 = 0; i0 < d; i0 += 64) {
        const uint64_t i = (uint64_t)i0 + lane;
        const uint32_t nu = i + 64 < d ? adj[i + 64] : 0;
        const bool in = i < d;
        const uint64_t V = __ballot(in);
        if (CHECK) {
            const uint32_t pu0 = (uint32_t)__shfl_up((int)cu, 1, 64), pu = lane ? pu0 : prev;
            if (__ballot(in && (cu >= n || (i > 0 && cu <= pu)))) return false;
        }
        const uint32_t top = lane_value(cu, 63);
        const uint32_t pn0 = (uint32_t)__shfl_up((int)nu, 1, 64);
        const uint64_t N = __ballot(i + 64 < d && nu == (lane ? pn0 : top) + 1);
        // T bit i: ids i - 1 .. i + 2 are consecutive
        const uint64_t C1 = (C >> 1) | (N << 63), T = C & C1 & ((C >> 2) | (N << 62));
        const uint64_t TN = N & (N >> 1) & (N >> 2) & 1;
        const uint64_t L = (T | (T << 1) | (TP >> 63) | (T << 2) | (TP >> 62) | (T >> 1) | (TN << 63)) & V;
        WaveChunk k;
        k.itv = L & ~C1;
        k.res = V & ~L;
        k.id = cu;
        const bool is_res = (k.res >> lane) & 1;
        const uint64_t mine = (is_res ? k.res : k.itv) & below;
        const uint32_t pv = (uint32_t)__shfl((int)cu, mine ? 63 - __builtin_clzll(mine) : 0, 64);
        const uint64_t open = ~C & ((2ull << lane) - 1);   // run starts up to this lane
        k.left = 0;
        k.len = 0;
        if (k.itv) {
            const uint32_t ls = (uint32_t)__shfl((int)cu, open ? 63 - __builtin_clzll(open) : 0, 64);
            k.left = open ? ls : run_left;
            k.len = cu - k.left + 1;
        }
        k.gap = is_res ? cu - (mine ? pv : last_res) - 1 : k.left - (mine ? pv + 1 : last_end) - 1;
        sink(k);
        const uint64_t st = ~C & V;
        if (st) run_left = lane_value(cu, 63 - __builtin_clzll(st));
        if (k.res) last_res = lane_value(cu, 63 - __builtin_clzll(k.res));
        if (k.itv) last_end = lane_value(cu, 63 - __builtin_clzll(k.itv)) + 1;
        prev = top;
        TP = T;
        C = N;
        cu = nu;
    }
    return true;
}

// Feeds a chunk's entries to the blocks.
template <class CloseI, class CloseR>
__device__ __forceinline__ void wave_feed(const WaveChunk &k, uint32_t v, WaveBlock &bi, WaveBlock &br, CloseI &&ci,
                                          CloseR &&cr) {
    const uint32_t lane = __lane_id();
    if (k.itv) {
        const bool e = (k.itv >> lane) & 1, first = bi.entries == 0 && (k.itv & ((1ull << lane) - 1)) == 0;
        const uint32_t lb = gamma_len32(k.len - MIN_RUN);
        bi.feed(k.itv, wave_scan(e && !first ? gamma_len32(k.gap) + lb : 0), e ? gamma_len32(nat32(k.left, v)) + lb : 0, ci);
    }
    if (k.res) {
        const bool e = (k.res >> lane) & 1, first = br.entries == 0 && (k.res & ((1ull << lane) - 1)) == 0;
        br.feed(k.res, wave_scan(e && !first ? zeta_len32(k.gap) : 0), e ? zeta_len32(nat32(k.id, v)) : 0, cr);
    }
}

template <bool CHECK>
__device__ __forceinline__ bool wave_plan(const uint32_t *__restrict__ adj, uint32_t d, uint32_t n, uint32_t v,
                                          WaveBlock &bi, WaveBlock &br) {
    return wave_row<CHECK>(adj, d, n, [&](const WaveChunk &k) {
        wave_feed(k, v, bi, br, [](uint32_t, uint32_t) {}, [](uint32_t, uint32_t) {});
    });
}

struct WaveRing {
    uint32_t iu[RING], ilen[RING], igap[RING];   // interval entries
    uint32_t ru[RING], rgap[RING];               // residual entries
    uint32_t seg[SEG_WORDS];                     // the segment being written
};

// ORs the low `len` bits (<= 64) of val into seg at bit `pos`, MSB first.
__device__ __forceinline__ void seg_or(uint32_t *seg, uint32_t pos, uint64_t val, uint32_t len) {
    const uint64_t x = val << (64 - len);
    const uint32_t w = pos >> 5, s = pos & 31;
    const uint64_t y = x >> s;
    const uint32_t a = (uint32_t)(y >> 32), b = (uint32_t)y, c = s ? (uint32_t)(x << (32 - s)) : 0u;
    if (a) atomicOr(&seg[w], a);
    if (b) atomicOr(&seg[w + 1], b);
    if (c) atomicOr(&seg[w + 2], c);
}

// Writes segment number k of a block (entries [s, e)) of the block at bit
// `start`; segment 0 takes the block's header along.
template <bool ITV>
__device__ __forceinline__ void wave_segment(WaveRing *R, uint64_t *words, uint64_t start, uint32_t segs, uint32_t k,
                                             uint32_t s, uint32_t e, uint32_t v) {
    const uint32_t lane = __lane_id();
    const uint32_t hl = gamma_len32(segs - 1);
    const uint64_t pos = start + (k ? hl + (uint64_t)SEG * k : 0);
    const uint32_t base = (uint32_t)(pos & 31);
    if (lane < SEG_WORDS) R->seg[lane] = 0;
    wave_sync();
    uint32_t off = base;
    const uint32_t cnt = e - s;
    if (k == 0) {
        if (lane == 0) seg_or(R->seg, off, segs, hl);
        off += hl;
    }
    if (lane == 0) seg_or(R->seg, off, (uint64_t)cnt + 1, gamma_len32(cnt));
    off += gamma_len32(cnt);
    for (uint32_t j0 = 0; j0 < cnt; j0 += 64) {
        const uint32_t j = j0 + lane, q = (s + j) & (RING - 1);
        const bool act = j < cnt;
        uint32_t c1 = 0, c2 = 0, l1 = 0, l2 = 0;
        if (act) {
            if (ITV) {
                c1 = j == 0 ? nat32(R->iu[q], v) : R->igap[q];
                c2 = R->ilen[q] - MIN_RUN;
                l1 = gamma_len32(c1);
                l2 = gamma_len32(c2);
            } else {
                c1 = j == 0 ? nat32(R->ru[q], v) : R->rgap[q];
                l1 = zeta_len32(c1);
            }
        }
        const uint32_t P = wave_scan(l1 + l2), o = off + P - l1 - l2;
        if (act) {
            if (ITV) {
                seg_or(R->seg, o, (uint64_t)c1 + 1, l1);
                seg_or(R->seg, o + l1, (uint64_t)c2 + 1, l2);
            } else {
                seg_or(R->seg, o, (1ull << (l1 / 4 * 3)) | ((uint64_t)c1 + 1), l1);
            }
        }
        off += lane_value(P, 63);
    }
    wave_sync();
    // stream word w (32 bits) is the high half of a 64-bit word when even
    uint32_t *out = reinterpret_cast<uint32_t *>(words);
    const uint64_t w0 = pos >> 5;
    const uint32_t nw = (off + 31) >> 5;
    if (lane < nw) {
        const uint32_t x = R->seg[lane];
        uint32_t *p = out + ((w0 + lane) ^ 1);
        if (lane == 0 || lane == nw - 1) {   // shared with the bits before and after
            if (x) atomicOr(p, x);
        } else {
            *p = x;
        }
    }
    wave_sync();
}

// Second pass over the row: the record's bits at `start` (words zeroed).
__device__ __forceinline__ void wave_write(WaveRing *R, uint64_t *words, uint64_t start, const uint32_t *__restrict__ adj,
                                           uint32_t d, uint32_t v, const WaveBlock &pi, const WaveBlock &pr) {
    const uint32_t lane = __lane_id();
    const uint64_t below = (1ull << lane) - 1;
    const uint32_t si = pi.segs(), sr = pr.segs();
    const uint64_t start_r = start + pi.bits();
    WaveBlock bi, br;
    // a closed segment is written when the next one closes: the last one
    // takes the tail
    uint32_t ki = 0, kr = 0;
    wave_row<false>(adj, d, 0, [&](const WaveChunk &k) {
        if ((k.itv >> lane) & 1) {
            const uint32_t q = (bi.entries + (uint32_t)__popcll(k.itv & below)) & (RING - 1);
            R->iu[q] = k.left;
            R->ilen[q] = k.len;
            R->igap[q] = k.gap;
        }
        if ((k.res >> lane) & 1) {
            const uint32_t q = (br.entries + (uint32_t)__popcll(k.res & below)) & (RING - 1);
            R->ru[q] = k.id;
            R->rgap[q] = k.gap;
        }
        wave_sync();
        wave_feed(k, v, bi, br,
                  [&](uint32_t s, uint32_t) {
                      if (bi.closed) wave_segment<true>(R, words, start, si, ki++, bi.last_idx, s, v);
                  },
                  [&](uint32_t s, uint32_t) {
                      if (br.closed) wave_segment<false>(R, words, start_r, sr, kr++, br.last_idx, s, v);
                  });
    });
    wave_segment<true>(R, words, start, si, si - 1, bi.tail_idx(), bi.entries, v);
    wave_segment<false>(R, words, start_r, sr, sr - 1, br.tail_idx(), br.entries, v);
}

}  // namespace enc

// Record lengths of the positions from `first` on whose rows have LANE_ROW < d
// <= long_min ids, a wave each; *err as k_encode_len.
__global__ void __launch_bounds__(64 * enc::ENC_WAVES) k_encode_wave_len(
    const uint64_t *__restrict__ row, const uint32_t *__restrict__ col, const uint32_t *__restrict__ vid,
    uint64_t first, uint64_t n_c, uint32_t n, uint64_t *__restrict__ len, unsigned long long *__restrict__ err, uint32_t long_min) {
    const uint64_t p = first + (uint64_t)blockIdx.x * enc::ENC_WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (p >= n_c) return;
    const uint32_t v = vid[p];
    const uint64_t r0 = row[v], r1 = row[v + 1];
    if (r1 < r0 || r1 - r0 <= enc::LANE_ROW || r1 - r0 > long_min) return;
    enc::WaveBlock bi, br;
    const bool ok = enc::wave_plan<true>(col + r0, (uint32_t)(r1 - r0), n, v, bi, br);
    if (__lane_id() == 0) {
        if (!ok) atomicCAS(err, 0ull, (unsigned long long)v + 1);
        len[p] = ok ? bi.bits() + br.bits() : 0;
    }
}

__global__ void __launch_bounds__(64 * enc::ENC_WAVES) k_encode_wave_write(
    const uint64_t *__restrict__ row, const uint32_t *__restrict__ col, const uint32_t *__restrict__ vid,
    uint64_t first, uint64_t n_c, const uint64_t *__restrict__ offs, uint64_t *words, uint32_t long_min) {
    __shared__ enc::WaveRing ring[enc::ENC_WAVES];
    const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint64_t p = first + (uint64_t)blockIdx.x * enc::ENC_WAVES + w;
    if (p >= n_c) return;
    const uint32_t v = vid[p];
    const uint64_t r0 = row[v], r1 = row[v + 1];
    if (r1 - r0 <= enc::LANE_ROW || r1 - r0 > long_min) return;
    enc::WaveBlock bi, br;
    (void)enc::wave_plan<false>(col + r0, (uint32_t)(r1 - r0), 0, v, bi, br);
    enc::wave_write(&ring[w], words, offs[p], col + r0, (uint32_t)(r1 - r0), v, bi, br);
}

}  // namespace lpa
