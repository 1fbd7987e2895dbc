// ytrc_k_vr_e.hip -- VolumeRenderSampler kernels: ColorTransferFunction with grey opacity.
#include "ytrc_kernels.h"
#include "ytrc_pick.h"

namespace ytrc {

// One field only; bit 1 is the n_samples == 10 unrolling, bit 3 a per-pixel lens.
pfn_t pick_persist_vr_e(int nfp, bool rec, int mode)
{
    if (nfp != 1) return nullptr;
    switch (mode) {
    case 33: return rec ? k_persist<1, 1, true, 33> : k_persist<1, 1, false, 33>;
    case 35: return rec ? k_persist<1, 1, true, 35> : k_persist<1, 1, false, 35>;
    case 41: return rec ? k_persist<1, 1, true, 41> : k_persist<1, 1, false, 41>;
    case 43: return rec ? k_persist<1, 1, true, 43> : k_persist<1, 1, false, 43>;
    default: return nullptr;
    }
}

kfn_t pick_kernel_vr_e(int nfp, bool rec, int mode)
{
    if (nfp != 1) return nullptr;
    switch (mode) {
    case 33: return rec ? k_render<1, 1, true, 33> : k_render<1, 1, false, 33>;
    case 35: return rec ? k_render<1, 1, true, 35> : k_render<1, 1, false, 35>;
    case 41: return rec ? k_render<1, 1, true, 41> : k_render<1, 1, false, 41>;
    case 43: return rec ? k_render<1, 1, true, 43> : k_render<1, 1, false, 43>;
    default: return nullptr;
    }
}

}  // namespace ytrc
