// Prefill GEMM instances: WF_I4T (bz_gemm.h).
#include "bz_gemm.h"

namespace bz {
int launch_gemm_i4t(const GemmParams& p, const GemmLaunch& l, hipStream_t st) { return launch_gemm_wf<WF_I4T>(p, l, st); }
}  // namespace bz
