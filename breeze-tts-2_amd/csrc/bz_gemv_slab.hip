// Instances of the few-row-block fp8 GEMV (bz_gemv_slab.h): the units per wave
// of the kernels it stands in for.
#include "bz_gemv_slab.h"

namespace bz {
int launch_slab(const StreamParams& p, const SlabLaunch& l, hipStream_t st) {
    switch (l.upw) {
        case 1: return launch_slab_kernel<1>(p, l, st);
        case 2: return launch_slab_kernel<2>(p, l, st);
        case 3: return launch_slab_kernel<3>(p, l, st);
        case 4: return launch_slab_kernel<4>(p, l, st);
        case 5: return launch_slab_kernel<5>(p, l, st);
        case 6: return launch_slab_kernel<6>(p, l, st);
        case 8: return launch_slab_kernel<8>(p, l, st);
        case 10: return launch_slab_kernel<10>(p, l, st);
        default: return BZ_ERR_INVALID_ARG;
    }
}
}  // namespace bz
