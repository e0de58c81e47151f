// Prefill GEMM instances: WF_F8T (bz_gemm.h).
#include "bz_gemm.h"

namespace bz {
int launch_gemm_f8t(const GemmParams& p, const GemmLaunch& l, hipStream_t st) { return launch_gemm_wf<WF_F8T>(p, l, st); }
}  // namespace bz
