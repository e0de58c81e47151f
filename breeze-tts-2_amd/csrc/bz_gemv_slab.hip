// Instances of the few-row-block fp8 GEMV (bz_gemv_slab.h).
#include "bz_gemv_slab.h"

namespace bz {
int launch_slab(const StreamParams& p, const SlabLaunch& l, hipStream_t st) {
    switch (l.m) {
        case 1: return launch_slab_rl<1>(p, l, st);
        case 2: return launch_slab_rl<2>(p, l, st);
        case 4: return launch_slab_rl<4>(p, l, st);
        default: return BZ_ERR_INVALID_ARG;
    }
}
}  // namespace bz
