// bins.hpp -- launches of the lane and group kernels (bins.hip): the bins of a
// step, and of the two-kernel method's decode.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "lp_kernels.hpp"

namespace lpa {

// A contiguous range of positions that one kernel handles.
struct Bin {
    int kind;          // LPA_BIN_*
    int param;         // LANE: network size N; WAVE/BLOCK: log2 table slots
    bool csr;          // small-vertex CSR part
    uint32_t begin, end;
};

// LDS bytes of the WAVE / BLOCK kernels' per-group table (2^logT slots) and
// neighbour list (2^logT / 2 ids), for ng groups per workgroup (the most that
// a launch takes).
inline size_t group_lds(int ng, uint32_t logT) { return (size_t)ng * 10ull * (1ull << logT); }
// groups per workgroup of a WAVE bin: a quarter wave per vertex up to
// quarter_max ids, a whole wave above
inline int wave_groups(uint32_t logT, uint32_t quarter_max = 128) {
    return (1u << (logT - 1)) <= quarter_max ? 16 : 4;
}

// label vectors staged per row gather by the group kernels: 8 from K = 5
// (one gather per neighbour and step at K = 8; with one aggregated match
// round the kernels stay fast enough at the lower occupancy that even label
// rows held by the 256 MB last-level cache gain from it), else K rounded
// down to 4 / 2 / 1.
inline int group_kb(uint32_t K) { return K >= 5 ? 8 : K >= 3 ? 4 : K == 2 ? 2 : 1; }

// Lanes per vertex of a WAVE bin, as groups per workgroup.  One or two
// vectors (8 staged ids per lane whatever the group): as few lanes as hold the
// list, 8 for up to 64 ids to 64 for 512, because a list of d ids is only
// about d / 20 segments to decode, a lane each.  More vectors: a quarter wave
// up to quarter_max ids, a wave above, and with 8 vectors per staged gather
// half waves above 64 ids (4 ids per lane up to 128) rather than quarter waves
// (8 per lane): half the staged registers, twice the waves resident.
// (quarter_max below 128 asks for whole waves above it, whatever K.)
inline int decode_groups(uint32_t logT) {
    const uint32_t cap = 1u << (logT - 1);
    return cap <= 64 ? 32 : cap <= 128 ? 16 : cap <= 256 ? 8 : 4;
}
inline int step_groups(uint32_t logT, uint32_t K, uint32_t quarter_max) {
    if (quarter_max == 0) quarter_max = 128;
    if (K <= 2 && quarter_max >= 128) return decode_groups(logT);
    const int ng = wave_groups(logT, quarter_max);
    return ng == 16 && (1u << (logT - 1)) > 64 && K >= 5 ? 8 : ng;
}
// dynamic LDS bytes of a bin's own launch, and of its part of a merged one
// (where the kernel's static LDS is dynamic too)
inline size_t step_lds(int ng, uint32_t logT, bool csr, uint32_t K) {
    const uint32_t cap = 1u << (logT - 1), G = BLOCK / ng, kb = group_kb(K);
    return (size_t)ng * 8 * group_words(group_list_inside(csr, K, kb, cap, staged_ids(kb, cap, G) * G), 1u << logT);
}
inline size_t static_bytes(size_t s) { return (s + 7) / 8 * 8; }
inline size_t merged_lds(int ng, uint32_t logT, bool csr, uint32_t K) {
    return step_lds(ng, logT, csr, K) +
           static_bytes(ng == 1 ? sizeof(GroupStatic<BLOCK, 8>) : ng == 4 ? sizeof(GroupStatic<64, 8>)
                        : ng == 8 ? sizeof(GroupStatic<32, 8>) : ng == 16 ? sizeof(GroupStatic<16, 8>)
                                                                          : sizeof(GroupStatic<8, 8>));
}
// whether the merged kernel has this bin's group kernel
inline bool merged(int ng, uint32_t logT, uint32_t K) {
    const uint32_t G = BLOCK / ng, kb = group_kb(K);
    return bins_hold(kb, G, staged_ids(kb, 1u << (logT - 1), G));
}

// Lets the kernels use `dyn` bytes of dynamic LDS (the device is current).
void bins_allow_lds(int dyn);
// One bin's positions [b.begin, b.end) by its own kernel; as_csr: rows from
// the CSR of `a`.
void launch_bin(const Bin &b, StepArgs a, bool as_csr, uint32_t quarter_max, hipStream_t s);
// LANE, WAVE and BLOCK bins of one step, all over the arguments `a`: bins too
// small to fill the device share a launch.  all_csr: every bin reads the CSR
// of `a`, else those of the small part do.
void launch_bins(const std::vector<Bin> &bins, const StepArgs &a, bool all_csr, uint32_t quarter_max, hipStream_t s);
// LANE, WAVE and BLOCK records decoded to CSR rows, likewise.
void launch_decode_bins(const std::vector<Bin> &bins, const DecodeArgs &a, hipStream_t s);

}  // namespace lpa
