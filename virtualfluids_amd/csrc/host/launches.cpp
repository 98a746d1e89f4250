// Sequences of launches: the entry points of a time step enqueued from a native loop.
#include "../vf_common.h"

extern "C" int vf_run_launches(const vf_launch* list, uint32_t n, uint32_t repeats, void* stream)
{
    using namespace vfa;
    if (n && !list) {
        set_last_error("run_launches: null list");
        return VF_ERR_INVALID_ARGUMENT;
    }
    for (uint32_t i = 0; i < n; ++i) {
        const vf_launch& l = list[i];
        const bool scaling = l.kind == VF_LAUNCH_COARSE_TO_FINE || l.kind == VF_LAUNCH_FINE_TO_COARSE;
        if (l.kind < VF_LAUNCH_BOX || l.kind > VF_LAUNCH_FINE_TO_COARSE || !l.level ||
            (l.kind == VF_LAUNCH_BC && !l.bc) || (scaling && !l.fine)) {
            set_last_error("run_launches: an entry of unknown kind, without a level, a launcher or a fine level");
            return VF_ERR_INVALID_ARGUMENT;
        }
    }
    for (uint32_t r = 0; r < repeats; ++r) {
        for (uint32_t i = 0; i < n; ++i) {
            const vf_launch& l = list[i];
            int rc = VF_OK;
            switch (l.kind) {
            case VF_LAUNCH_BOX: rc = vf_k17_run_box(l.level, l.collisionTemplate, stream); break;
            case VF_LAUNCH_BOX_BOUNCE_BACK:
                rc = vf_k17_run_box_bounce_back(l.level, l.collisionTemplate, l.bounceBack, stream);
                break;
            case VF_LAUNCH_INDICES:
                rc = vf_k17_run_on_indices(l.level, l.level->fluidNodeIndices, l.level->numberOfFluidNodes,
                                           l.collisionTemplate, stream);
                break;
            case VF_LAUNCH_BC: rc = l.bc(l.level, l.list, stream); break;
            case VF_LAUNCH_SWAP: l.level->isEvenTimestep = l.level->isEvenTimestep ? 0 : 1; break;
            case VF_LAUNCH_COARSE_TO_FINE:
                rc = vf_ScaleCoarseToFineCompressible(l.level, l.fine, l.cells, l.offsets, stream);
                break;
            default: rc = vf_ScaleFineToCoarseCompressible(l.level, l.fine, l.cells, l.offsets, stream); break;
            }
            if (rc != VF_OK) return rc;
        }
    }
    return VF_OK;
}
