// cgr_decode.hpp -- device-side CGR bit reader and segment decoders (gfx950).
//
// Restates the reference's CgrReader / IntervalSegmentHelper /
// ResidualSegmentHelper (include/graph_utils.cuh:19-183) for 64-bit
// windows: the stream is held as 64-bit words whose bit order is the
// stream order (bit 0 of the stream is the MSB of word 0), every code of a
// graph with n < 2^30 fits one 64-bit window, and bit offsets are 64-bit
// (the reference's 32-bit global_offset overflows beyond 2^32 bits,
// graph_utils.cuh:22).  A reader keeps a 6-word register window per segment.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// The reader and the serial decoders also build for the host, where a test
// library checks them against the CPU oracle.
#define LPA_HD __host__ __device__

namespace lpa {

constexpr uint32_t SEG_BITS = 256;   // segment stride (graph_utils.cuh:17)
constexpr uint32_t MIN_ITV = 4;      // interval length offset (graph_utils.cuh:172)

struct BitReader {
    // Six words are loaded together at every seek (one memory latency per
    // 256-bit segment); moving to the next word shifts the registers down
    // without a load, and only a segment longer than ~320 bits (the merged
    // last segment of a block) triggers a second batch.  A reader that
    // loaded the next word at every word step would stall on that load at
    // the step itself (the shifted-in value is copied immediately).
    static constexpr int NW = 6;
    const uint64_t *__restrict__ W;
    uint64_t pos;     // absolute bit position
    uint64_t idx;     // word index held in w[0]
    uint32_t left;    // valid words from w[0]
    uint64_t w[NW];

    LPA_HD __forceinline__ void load_at(uint64_t i) {
#pragma unroll
        for (int k = 0; k < NW; k++) w[k] = W[i + k];
        idx = i;
        left = NW;
    }
    LPA_HD __forceinline__ void seek(const uint64_t *__restrict__ words, uint64_t p) {
        W = words;
        pos = p;
        load_at(p >> 6);
    }
    // Moves forward to bit q >= pos: by shifting when q lies in the loaded
    // words, else by a new batch load.
    LPA_HD __forceinline__ void move_to(uint64_t q) {
        const uint64_t d = (q >> 6) - idx;
        if (d + 2 <= left) {
#pragma unroll
            for (int step = 1; step < NW - 1; step++) {
                if ((uint64_t)step > d) break;
#pragma unroll
                for (int k = 0; k < NW - 1; k++) w[k] = w[k + 1];
            }
            idx += d;
            left -= (uint32_t)d;
            pos = q;
        } else {
            pos = q;
            load_at(q >> 6);
        }
    }
    // 64 bits starting at pos; pos - idx*64 < 64 always holds.
    LPA_HD __forceinline__ uint64_t window() const {
        uint32_t s = (uint32_t)(pos & 63);
        return s ? (w[0] << s) | (w[1] >> (64 - s)) : w[0];
    }
    LPA_HD __forceinline__ void advance(uint32_t bits) {
        pos += bits;
        if ((pos >> 6) != idx) {   // codes are < 64 bits: at most one word step
#pragma unroll
            for (int k = 0; k < NW - 1; k++) w[k] = w[k + 1];
            idx++;
            if (--left < 2) load_at(idx);
        }
    }
    // Elias gamma: 0^L then the L+1 bits of x+1 (graph_utils.cuh:63-67)
    LPA_HD __forceinline__ uint32_t gamma() {
        uint64_t x = window();
        uint32_t L = (uint32_t)__builtin_clzll(x | 1ull);   // L <= 31 for n < 2^30
        uint32_t len = 2 * L + 1;
        uint64_t y = x >> (64 - len);
        advance(len);
        return (uint32_t)(y - 1);
    }
    // zeta_3: 0^h 1 then 3(h+1) bits of x+1 (graph_utils.cuh:70-77)
    LPA_HD __forceinline__ uint32_t zeta() {
        uint64_t x = window();
        uint32_t h = (uint32_t)__builtin_clzll(x | 1ull);
        uint32_t body = 3 * (h + 1);
        uint64_t y = (x << (h + 1)) >> (64 - body);
        advance(4 * (h + 1));
        return (uint32_t)(y - 1);
    }
};

// Reader over a range of the stream staged as 32-bit words in LDS (stream
// order, MSB first; word k of the range at w[k + 2], so that every position
// has a word before it).  q = bit position in the range + 63: with s = (q & 31)
// + 1 bits of w[q >> 5] consumed, the 32 bits at the position are one funnel
// shift of two words, for any alignment.  Nearly every code is at most 32
// bits long (gamma below 2^16 - 1, zeta_3 below 2^24 - 1) and costs a dozen
// 32-bit instructions and one LDS read; longer ones take a third word.
// BitReader's 64-bit shifts and its shifting of six words cost several times
// that.  R-MAT 20, K = 1, settled steps: group kernels of 16 / 64 / 256 lanes
// 28.5 / 56.6 / 44.9 -> 22.4 / 48.1 / 40.7 us per launch; R-MAT 19 decoded to
// CSR with coalesced stores besides: 316 -> 160 us per step.
// CHECK: words from index `lim` on are not staged and are read from the
// stream itself (64-bit words W from index `base`).
template <bool CHECK> struct WinReader {
    const uint32_t *w;
    uint32_t q;
    uint32_t lim;
    const uint64_t *__restrict__ W;
    uint64_t base;

    LPA_HD __forceinline__ void set(uint64_t bit) { q = (uint32_t)(bit - (base << 6)) + 63; }
    LPA_HD __forceinline__ uint32_t stream_word(uint32_t k) const {
        const uint64_t x = W[base + ((k - 2) >> 1)];
        return (k & 1) ? (uint32_t)x : (uint32_t)(x >> 32);
    }
    static LPA_HD __forceinline__ uint32_t funnel(uint32_t a, uint32_t b, uint32_t q) {
#ifdef __HIP_DEVICE_COMPILE__
        return __builtin_amdgcn_alignbit(a, b, ~q);   // by the low 5 bits of ~q
#else
        return (uint32_t)((((uint64_t)a << 32) | b) >> (~q & 31));
#endif
    }
    LPA_HD __forceinline__ uint32_t window() const {
        const uint32_t k = q >> 5;
        uint32_t a, b;
        if (!CHECK || k + 1 < lim) {
            a = w[k];
            b = w[k + 1];
        } else {
            a = stream_word(k);
            b = stream_word(k + 1);
        }
        return funnel(a, b, q);
    }
    // 64 bits at the position, `hi` its first 32
    LPA_HD __forceinline__ uint64_t window64(uint32_t hi) const {
        const uint32_t k = q >> 5;
        uint32_t b, c;
        if (!CHECK || k + 2 < lim) {
            b = w[k + 1];
            c = w[k + 2];
        } else {
            b = stream_word(k + 1);
            c = stream_word(k + 2);
        }
        return ((uint64_t)hi << 32) | funnel(b, c, q);
    }
    LPA_HD __forceinline__ uint32_t gamma() {
        const uint32_t hi = window();
        if (hi >> 16) {
            const uint32_t L = (uint32_t)__builtin_clz(hi), y = hi >> (31 - 2 * L);
            q += 2 * L + 1;
            return y - 1;
        }
        const uint64_t x = window64(hi);
        const uint32_t L = (uint32_t)__builtin_clzll(x | 1ull), len = 2 * L + 1;
        q += len;
        return (uint32_t)((x >> (64 - len)) - 1);
    }
    LPA_HD __forceinline__ uint32_t zeta() {
        const uint32_t hi = window();
        if (hi >> 24) {
            const uint32_t h = (uint32_t)__builtin_clz(hi);
            const uint32_t y = (hi << (h + 1)) >> (29 - 3 * h);
            q += 4 * h + 4;
            return y - 1;
        }
        const uint64_t x = window64(hi);
        const uint32_t h = (uint32_t)__builtin_clzll(x | 1ull), body = 3 * (h + 1);
        q += 4 * (h + 1);
        return (uint32_t)(((x << (h + 1)) >> (64 - body)) - 1);
    }
};

// Stream word pair as staged: the 32 bits that come first at the lower index.
LPA_HD __forceinline__ uint64_t staged_pair(uint64_t x) { return (x >> 32) | (x << 32); }

// decode_first_num (graph_utils.cuh:34-37)
LPA_HD __forceinline__ uint32_t from_nat(uint32_t v, uint32_t x) {
    return (x & 1) ? v - (x >> 1) - 1 : v + (x >> 1);
}

// Decodes the interval segment the reader stands at (vertex v); calls
// emit_run(left, len) for every interval; leaves the reader after it.
template <class R, class F>
LPA_HD __forceinline__ void read_interval_segment(R &r, uint32_t v, F &&emit_run) {
    const uint32_t c = r.gamma();
    uint32_t stop = 0;
    for (uint32_t t = 0; t < c; t++) {
        const uint32_t left = (t == 0) ? from_nat(v, r.gamma()) : stop + r.gamma() + 1;
        const uint32_t len = r.gamma() + MIN_ITV;
        emit_run(left, len);
        stop = left + len;
    }
}

// Decodes the c ids of a residual segment (the reader stands after its count).
template <class R, class F>
LPA_HD __forceinline__ void read_residual_ids(R &r, uint32_t v, uint32_t c, F &&emit) {
    if (c == 0) return;
    uint32_t cur = from_nat(v, r.zeta());
    emit(cur);
    for (uint32_t t = 1; t < c; t++) {
        cur += r.zeta() + 1;
        emit(cur);
    }
}

// Decodes the residual segment the reader stands at; emit(u) per neighbour.
template <class R, class F>
LPA_HD __forceinline__ void read_residual_segment(R &r, uint32_t v, F &&emit) {
    const uint32_t c = r.gamma();
    read_residual_ids(r, v, c, emit);
}

// Serial decode of a whole staged record (the reader stands at its start):
// emit(u) per neighbour, in encoded order.
template <class R, class F>
LPA_HD __forceinline__ void read_record(R &r, uint32_t v, F &&emit) {
    uint32_t ns = r.gamma() + 1, base = r.q;
    for (uint32_t j = 0; j < ns; j++) {
        r.q = base + SEG_BITS * j;
        read_interval_segment(r, v, [&](uint32_t l, uint32_t len) {
            for (uint32_t x = 0; x < len; x++) emit(l + x);
        });
    }
    ns = r.gamma() + 1;
    base = r.q;
    for (uint32_t j = 0; j < ns; j++) {
        r.q = base + SEG_BITS * j;
        read_residual_segment(r, v, emit);
    }
}

// Serial decode of a whole record by one lane with one reader: emit(u) per
// neighbour, in encoded order (intervals, then residuals).  Padded segments
// are reached by shifting the loaded words when they are close.  Returns
// the bit after the record.
template <class F>
LPA_HD __forceinline__ uint64_t decode_record(const uint64_t *__restrict__ W, uint64_t p, uint32_t v,
                                                  F &&emit) {
    BitReader r;
    r.seek(W, p);
    uint32_t ns = r.gamma() + 1;
    uint64_t base = r.pos;
    for (uint32_t j = 0; j < ns; j++) {
        r.move_to(base + (uint64_t)SEG_BITS * j);
        read_interval_segment(r, v, [&](uint32_t l, uint32_t len) {
            for (uint32_t x = 0; x < len; x++) emit(l + x);
        });
    }
    ns = r.gamma() + 1;
    base = r.pos;
    for (uint32_t j = 0; j < ns; j++) {
        r.move_to(base + (uint64_t)SEG_BITS * j);
        read_residual_segment(r, v, emit);
    }
    return r.pos;
}

}  // namespace lpa
