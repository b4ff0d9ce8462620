// bins.hip -- the lane and group kernels and their launches (see bins.hpp).
#include "bins.hpp"

#include <algorithm>

#include "lpa_amd.h"

namespace lpa {

__global__ void __launch_bounds__(BLOCK) k_decode_bins(DecodeArgs a, BinTable t) {
    extern __shared__ uint64_t lds[];
    uint32_t i = 0;
    while (i + 1 < t.n && blockIdx.x >= t.e[i + 1].first) i++;
    const BinTable::Entry e = t.e[i];
    decode_bin(a, e, blockIdx.x - e.first, lds);
}

template <bool CSR> static void launch_lane(int N, StepArgs a, uint32_t count, hipStream_t s) {
    dim3 grid((count + BLOCK - 1) / BLOCK);
    switch (N) {
    case 4: hipLaunchKernelGGL((k_lane<4, CSR>), grid, dim3(BLOCK), 0, s, a); break;
    case 8: hipLaunchKernelGGL((k_lane<8, CSR>), grid, dim3(BLOCK), 0, s, a); break;
    case 16: hipLaunchKernelGGL((k_lane<16, CSR>), grid, dim3(BLOCK), 0, s, a); break;
    case 32: hipLaunchKernelGGL((k_lane<32, CSR>), grid, dim3(BLOCK), 0, s, a); break;
    default: hipLaunchKernelGGL((k_lane<64, CSR>), grid, dim3(BLOCK), 0, s, a); break;
    }
}

// instance of the group kernel for a batch size and staged ids per lane
template <int G, bool CSR> static const void *group_fn(int kb, uint32_t ids) {
    switch (kb) {
    case 1: return (const void *)k_group<G, CSR, 1, 8>;
    case 2: return (const void *)k_group<G, CSR, 2, 8>;
    case 4:
        return ids == 2 ? (const void *)k_group<G, CSR, 4, 2>
             : ids == 4 ? (const void *)k_group<G, CSR, 4, 4> : (const void *)k_group<G, CSR, 4, 8>;
    default:
        return ids == 2 ? (const void *)k_group<G, CSR, 8, 2>
             : ids == 4 ? (const void *)k_group<G, CSR, 8, 4> : (const void *)k_group<G, CSR, 8, 8>;
    }
}

template <int G>
static void launch_group(bool as_csr, dim3 grid, size_t lds, hipStream_t s, const StepArgs &a, uint32_t logT,
                         uint32_t cap) {
    const int kb = group_kb(a.K);
    const uint32_t ids = staged_ids(kb, cap, G);
    const void *fn = as_csr ? group_fn<G, true>(kb, ids) : group_fn<G, false>(kb, ids);
    StepArgs args = a;
    void *params[] = {&args, &logT, &cap};
    (void)hipLaunchKernel(fn, grid, dim3(BLOCK), params, lds, s);
}

template <int G> static void allow_group_lds(int dyn) {
    for (int kb : {1, 2, 4, 8})
        for (uint32_t ids : {2u, 4u, 8u})
            for (const void *f : {group_fn<G, false>(kb, ids), group_fn<G, true>(kb, ids)})
                (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, dyn);
}

// k_bins<KB> (bins_merged.hip)
const void *bins_fn_1();
const void *bins_fn_2();
const void *bins_fn_4();
const void *bins_fn_8();
static const void *bins_fn(uint32_t K) {
    switch (group_kb(K)) {
    case 1: return bins_fn_1();
    case 2: return bins_fn_2();
    case 4: return bins_fn_4();
    default: return bins_fn_8();
    }
}

void bins_allow_lds(int dyn) {
    allow_group_lds<8>(dyn);
    allow_group_lds<16>(dyn);
    allow_group_lds<32>(dyn);
    allow_group_lds<64>(dyn);
    allow_group_lds<BLOCK>(dyn);
    for (const void *f : {bins_fn(1), bins_fn(2), bins_fn(4), bins_fn(8), (const void *)k_decode_bins})
        (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, dyn);
}

void launch_bin(const Bin &b, StepArgs a, bool as_csr, uint32_t quarter_max, hipStream_t s) {
    a.begin = b.begin;
    a.end = b.end;
    const uint32_t count = b.end - b.begin;
    if (count == 0) return;
    const uint32_t logT = (uint32_t)b.param, cap = logT ? 1u << (logT - 1) : 0;
    switch (b.kind) {
    case LPA_BIN_LANE:
        if (as_csr) launch_lane<true>(b.param, a, count, s);
        else launch_lane<false>(b.param, a, count, s);
        break;
    case LPA_BIN_WAVE: {
        const int ng = step_groups(logT, a.K, quarter_max);
        const size_t lds = step_lds(ng, logT, as_csr, a.K);
        const dim3 grid((count + ng - 1) / ng);
        if (ng == 32) launch_group<8>(as_csr, grid, lds, s, a, logT, cap);
        else if (ng == 16) launch_group<16>(as_csr, grid, lds, s, a, logT, cap);
        else if (ng == 8) launch_group<32>(as_csr, grid, lds, s, a, logT, cap);
        else launch_group<64>(as_csr, grid, lds, s, a, logT, cap);
        break;
    }
    case LPA_BIN_BLOCK: launch_group<BLOCK>(as_csr, dim3(count), step_lds(1, logT, as_csr, a.K), s, a, logT, cap); break;
    default: break;   // heavy bins run through their own kernels
    }
}

// Workgroups up to which a bin shares its launch with other small ones: with
// the LDS of the largest (up to 50 KB), three to four workgroups fit a CU, so
// about this many run at once (4096: 3 to 5 % slower on R-MAT 19 and 20, all in
// one 9 % slower).  20 steps of R-MAT 12 2.71 -> 1.42 ms (a step
// of 13 launches -> 4), R-MAT 20 K = 1 10.0 -> 9.0, R-MAT 19 two-kernel 8.3 ->
// 6.9, R-MAT 17 K = 64 44.7 -> 34.2, copying graphs 6.9 -> 5.5 (K = 1) and 10.6 ->
// 6.9 ms (K = 5).
constexpr uint32_t MERGE_BLOCKS = 1024;

// Table entries of several launches; the most demanding bins first, so that
// the last workgroups to start are short ones.
struct Merge {
    BinTable t{};
    uint32_t blocks = 0;
    size_t lds = 0;
    void add(const Bin &b, uint32_t code, bool csr, uint32_t logT, uint32_t wg, size_t bytes) {
        t.e[t.n++] = {blocks, b.begin, b.end, code, csr ? 1u : 0u, logT};
        blocks += wg;
        lds = std::max(lds, bytes);
    }
};

static uint32_t group_code(int ng) {
    return ng == 1 ? BC_G256 : ng == 4 ? BC_G64 : ng == 8 ? BC_G32 : ng == 16 ? BC_G16 : BC_G8;
}

template <int N> static size_t lane_bytes(bool csr) {
    return csr ? sizeof(LaneShared<N, true>) : sizeof(LaneShared<N, false>);
}

void launch_bins(const std::vector<Bin> &bins, const StepArgs &a, bool all_csr, uint32_t quarter_max, hipStream_t s) {
    Merge m;
    const Bin *last = nullptr;
    auto flush = [&] {
        if (m.t.n == 1) {
            launch_bin(*last, a, all_csr || last->csr, quarter_max, s);
        } else if (m.t.n) {
            StepArgs args = a;
            void *params[] = {&args, &m.t};
            (void)hipLaunchKernel(bins_fn(a.K), dim3(m.blocks), dim3(BLOCK), params, m.lds, s);
        }
        m = Merge{};
    };
    for (auto it = bins.rbegin(); it != bins.rend(); ++it) {
        const Bin &b = *it;
        const uint32_t count = b.end - b.begin, logT = (uint32_t)b.param;
        if (count == 0) continue;
        uint32_t code, wg;
        size_t bytes;
        bool held = true;
        const bool csr = all_csr || b.csr;
        if (b.kind == LPA_BIN_LANE) {
            wg = (count + BLOCK - 1) / BLOCK;
            switch (b.param) {
            case 4: code = BC_LANE4; bytes = lane_bytes<4>(csr); break;
            case 8: code = BC_LANE8; bytes = lane_bytes<8>(csr); break;
            case 16: code = BC_LANE16; bytes = lane_bytes<16>(csr); break;
            case 32: code = BC_LANE32; bytes = lane_bytes<32>(csr); break;
            default: code = BC_LANE64; bytes = 0; held = false; break;
            }
        } else if (b.kind == LPA_BIN_WAVE || b.kind == LPA_BIN_BLOCK) {
            const int ng = b.kind == LPA_BIN_BLOCK ? 1 : step_groups(logT, a.K, quarter_max);
            wg = (count + ng - 1) / ng;
            code = group_code(ng);
            bytes = merged_lds(ng, logT, csr, a.K);
            held = merged(ng, logT, a.K);
        } else {
            continue;
        }
        // the XCD mapping is per launch, and the recorder times whole bins
        if (wg > MERGE_BLOCKS || !held || a.xcds > 1 || a.rec) {
            launch_bin(b, a, csr, quarter_max, s);
            continue;
        }
        if (m.t.n == BinTable::MAX) flush();
        last = &b;
        m.add(b, code, csr, logT, wg, bytes);
    }
    flush();
}

void launch_decode_bins(const std::vector<Bin> &bins, const DecodeArgs &a, hipStream_t s) {
    Merge m;
    auto flush = [&] {
        if (m.t.n) hipLaunchKernelGGL(k_decode_bins, dim3(m.blocks), dim3(BLOCK), m.lds, s, a, m.t);
        m = Merge{};
    };
    for (auto it = bins.rbegin(); it != bins.rend(); ++it) {
        const Bin &b = *it;
        const uint32_t count = b.end - b.begin, logT = (uint32_t)b.param;
        if (count == 0) continue;
        Merge one;
        if (b.kind == LPA_BIN_LANE) {
            const uint32_t wg = (count + BLOCK - 1) / BLOCK;
            switch (b.param) {
            case 4: one.add(b, BC_LANE4, false, 0, wg, sizeof(LaneDecodeShared<4>)); break;
            case 8: one.add(b, BC_LANE8, false, 0, wg, sizeof(LaneDecodeShared<8>)); break;
            case 16: one.add(b, BC_LANE16, false, 0, wg, sizeof(LaneDecodeShared<16>)); break;
            case 32: one.add(b, BC_LANE32, false, 0, wg, sizeof(LaneDecodeShared<32>)); break;
            default: one.add(b, BC_LANE64, false, 0, wg, sizeof(LaneDecodeShared<64>)); break;
            }
        } else if (b.kind == LPA_BIN_WAVE || b.kind == LPA_BIN_BLOCK) {
            const int ng = b.kind == LPA_BIN_BLOCK ? 1 : decode_groups(logT);
            const size_t st = ng == 1 ? sizeof(GroupDecodeStatic<BLOCK>) : ng == 4 ? sizeof(GroupDecodeStatic<64>)
                              : ng == 8 ? sizeof(GroupDecodeStatic<32>) : ng == 16 ? sizeof(GroupDecodeStatic<16>)
                                                                                   : sizeof(GroupDecodeStatic<8>);
            one.add(b, group_code(ng), false, logT, (count + ng - 1) / ng, (size_t)ng * 6ull * (1ull << logT) + static_bytes(st));
        } else {
            continue;
        }
        if (one.blocks > MERGE_BLOCKS) {
            hipLaunchKernelGGL(k_decode_bins, dim3(one.blocks), dim3(BLOCK), one.lds, s, a, one.t);
            continue;
        }
        if (m.t.n == BinTable::MAX) flush();
        const BinTable::Entry &e = one.t.e[0];
        m.add(b, e.code, false, e.logT, one.blocks, one.lds);
    }
    flush();
}

}  // namespace lpa
