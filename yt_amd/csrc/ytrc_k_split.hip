// ytrc_k_split.hip -- volume renders of few tiles: four waves to a tile.
#include "ytrc_kernels.h"
#include "ytrc_pick.h"

namespace ytrc {

// One field, no record, ColorTransferFunction in transmittance form: bit 1
// is the n_samples == 10 unrolling, bit 3 a per-pixel lens.
pfn_t pick_split(int kind, int mode)
{
    if (kind != 1) return nullptr;
    switch (mode) {
    case 1: return k_split<1>;
    case 3: return k_split<3>;
    case 9: return k_split<9>;
    case 11: return k_split<11>;
    default: return nullptr;
    }
}

}  // namespace ytrc
