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
    uint32_t maxdeg;
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
