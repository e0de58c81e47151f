// Instances of the bf16 decode GEMV (bz_gemv_rows.h).
#include "bz_gemv_rows.h"

namespace bz {
int launch_rows(const GemvParams& p, const RowsLaunch& l, int rows, hipStream_t st) {
    switch (l.m) {
        case 1: return launch_rows_kc<1>(p, l, rows, st);
        case 2: return launch_rows_kc<2>(p, l, rows, st);
        case 4: return launch_rows_kc<4>(p, l, rows, st);
        default: return BZ_ERR_INVALID_ARG;
    }
}
}  // namespace bz
