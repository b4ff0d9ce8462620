// bins_merged.hip -- the kernel of several bins at once, for batches of
// BINS_KB label vectors (compiled once per batch size: 1, 2, 4, 8).
#include "lp_kernels.hpp"

#define BINS_NAME2(kb) bins_fn_##kb
#define BINS_NAME(kb) BINS_NAME2(kb)

namespace lpa {
const void *BINS_NAME(BINS_KB)() { return (const void *)k_bins<BINS_KB>; }
}  // namespace lpa
