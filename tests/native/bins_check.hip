// bins_check.hip -- test library: the LDS that a launch of the group kernels
// is given (bins.hpp) and the LDS that the kernel it reaches addresses
// (lp_kernels.hpp), as plain host arithmetic.
#include "../../lpa_amd/csrc/hip/bins.hpp"

using namespace lpa;

namespace {
// Bytes that group_tile<G, CSR, KB, IPL> addresses over a list of cap ids.
size_t tile_bytes(uint32_t G, bool csr, uint32_t KB, uint32_t IPL, uint32_t K, uint32_t logT) {
    const uint32_t cap = 1u << (logT - 1), ng = BLOCK / G;
    const bool inside = group_list_inside(csr, K, KB, cap, IPL * G);
    // CSR rows need no list; a list inside takes the table's upper half
    const size_t list = csr ? 0 : inside ? 0 : (size_t)cap * 4;
    const size_t last = (size_t)(ng - 1) * group_words(inside, 1u << logT) * 8;
    return last + ((size_t)8 << logT) + list;
}
template <int G> size_t static_of(uint32_t KB) {
    return KB == 1 ? sizeof(GroupStatic<G, 1>) : KB == 2 ? sizeof(GroupStatic<G, 2>)
         : KB == 4 ? sizeof(GroupStatic<G, 4>) : sizeof(GroupStatic<G, 8>);
}
}  // namespace

extern "C" {

// block: a BLOCK bin, else a WAVE bin.  out: groups, IPL of the separate
// launch, bytes it gets, bytes it addresses, whether the bin may be merged,
// bytes it adds up to there, bytes it addresses there.
void bc_plan(uint32_t K, uint32_t quarter_max, uint32_t logT, int block, int csr, uint64_t *out) {
    const int ng = block ? 1 : step_groups(logT, K, quarter_max);
    const uint32_t G = BLOCK / ng, kb = group_kb(K), cap = 1u << (logT - 1), ids = staged_ids(kb, cap, G);
    out[0] = ng;
    out[1] = ids;
    out[2] = step_lds(ng, logT, csr, K);
    out[3] = tile_bytes(G, csr, kb, ids, K, logT);
    out[4] = merged(ng, logT, K);
    out[5] = merged_lds(ng, logT, csr, K);
    const size_t st = G == 8 ? static_of<8>(kb) : G == 16 ? static_of<16>(kb) : G == 32 ? static_of<32>(kb)
                    : G == 64 ? static_of<64>(kb) : static_of<BLOCK>(kb);
    out[6] = (st + 7) / 8 * 8 + tile_bytes(G, csr, kb, ids, K, logT);
}

// Whether k_bins<kb> of a bin with these groups and staged ids does anything.
int bc_held(uint32_t kb, uint32_t G, uint32_t ids) { return bins_hold(kb, G, ids); }

}  // extern "C"
