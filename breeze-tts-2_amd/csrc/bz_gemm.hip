// Host side of the prefill GEMM (C ABI entries bz_gemm_tiled and
// bz_gemm_workspace) and the sum over its K slices.
#include <algorithm>

#include "bz_gemm.h"

namespace bz {


// Sums of the K slices in slice order, four columns per thread.
__global__ void __launch_bounds__(256) gemm_sum_slices(const float* part, int nsl, int M, int N, void* out, int64_t ldo,
                                                       int out_f32) {
    const int64_t item = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int nq = N >> 2;
    if (item >= (int64_t)M * nq) return;
    const int m = (int)(item / nq), c = (int)(item - (int64_t)m * nq) * 4;
    const int64_t stride = (int64_t)M * N;
    const float* s = part + (int64_t)m * N + c;
    f32x4_t a = *reinterpret_cast<const f32x4_t*>(s);
    for (int i = 1; i < nsl; ++i) a += *reinterpret_cast<const f32x4_t*>(s + i * stride);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (out_f32)
            static_cast<float*>(out)[(int64_t)m * ldo + c + q] = a[q];
        else
            static_cast<uint16_t*>(out)[(int64_t)m * ldo + c + q] = f32_to_bf16(a[q]);
    }
}

struct GemmPlan {
    GemmLaunch l;
    int mtiles, ntiles, nsl, sps;
    size_t ws;
};

// Microseconds a launch shape is expected to take, from which the rule picks
// the smallest.  Fitted to graph replays over 88 (M, N, K) per format on
// MI355X (M = 33..2048; the model's layer shapes and 1024..10240 squared
// ones), about 4900 timings: one workgroup's steps of 256 k, plus its start
// and epilogue, times the rounds of 256 CUs the grid needs (tiles of up to 8
// groups x blocks fit a CU twice, so their rounds overlap), plus the second
// launch and its traffic where K is sliced.  Over those shapes the shape it
// picks takes 2% (int4) / 3% (fp8) longer than the best of the sweep on
// average, at worst 24% / 42% (fp8 K2048 N6144 M = 256: 23.9 us for 16.8).
struct GemmCost {
    float step0, step_m, step_n, step_mn, wg0, wg_mn, overlap, sum0, sum_mb, traffic_mb;
};
constexpr GemmCost kGemmCostI4 = {-0.245f, 0.144f, 0.374f, 0.0156f, -0.457f, 0.154f, 0.546f, 1.90f, 1.89f, 0.0106f};
constexpr GemmCost kGemmCostF8 = {-0.206f, 0.108f, 0.217f, 0.0215f, 0.365f, 0.210f, 0.547f, 1.60f, 1.57f, 0.0172f};

static float gemm_cost(int wf, int M, int N, int K, int mt, int nt, const GemmPlan& pl) {
    const GemmCost& c = tiled_i4(wf) ? kGemmCostI4 : kGemmCostF8;
    const float mn = (float)(mt * nt);
    const float one = c.wg0 + c.wg_mn * mn +
                      (float)(pl.sps + (pl.sps & 1)) * (c.step0 + c.step_m * mt + c.step_n * nt + c.step_mn * mn);
    const float full = (float)pl.l.grid / 256.0f;
    const float rounds = mn > 8.0f ? (float)((pl.l.grid + 255) / 256) : full <= 1.0f ? 1.0f : full + c.overlap;
    const float w_mb = (float)N * (float)K * (tiled_i4(wf) ? 0.53e-6f : 1e-6f), x_mb = (float)M * (float)K * 2e-6f;
    const float sums = pl.nsl > 1 ? c.sum0 + c.sum_mb * (float)pl.nsl * (float)M * (float)N * 1e-6f : 0.0f;
    return one * rounds + sums + c.traffic_mb * ((float)pl.mtiles * w_mb + (float)pl.ntiles * x_mb);
}

// The plan of one launch shape; nsl is lowered to the slices that get steps.
static int gemm_shape(int M, int N, int K, int mt, int nt, int nsl, GemmPlan& pl) {
    const int steps = (K + kGemmStepK - 1) / kGemmStepK, nblk = N / 16;
    pl.l.mt = mt;
    pl.l.nt = nt;
    pl.mtiles = (M + mt * 16 - 1) / (mt * 16);
    pl.ntiles = (nblk + kGemmColWaves * nt - 1) / (kGemmColWaves * nt);
    nsl = std::min(nsl, steps);
    pl.sps = (steps + nsl - 1) / nsl;
    pl.nsl = (steps + pl.sps - 1) / pl.sps;
    const int64_t grid = (int64_t)pl.mtiles * pl.ntiles * pl.nsl;
    if (grid > 0x7FFFFFFF) return BZ_ERR_UNSUPPORTED;
    pl.l.grid = (unsigned)grid;
    pl.ws = pl.nsl > 1 ? (size_t)pl.nsl * M * N * 4 : 0;
    return BZ_OK;
}

// K slices only where the grid stays within about two rounds: more of them
// never won a timing.
constexpr int kGemmSlices[] = {1, 2, 3, 4, 6, 8, 12};
constexpr unsigned kGemmSlicedGrid = 520;

static int gemm_plan(int wf, int M, int N, int K, int cfg_mt, int cfg_nt, int cfg_nsl, GemmPlan& pl) {
    if (cfg_nsl > 64) return BZ_ERR_INVALID_ARG;
    float best = 0.0f;
    bool found = false;
    for (int mt : kGemmMt)
        for (int nt : kGemmNt) {
            if (!gemm_shape_ok(mt, nt) || (cfg_mt && cfg_mt != mt) || (cfg_nt && cfg_nt != nt)) continue;
            for (int nsl : kGemmSlices) {
                GemmPlan q;
                const int rc = gemm_shape(M, N, K, mt, nt, cfg_nsl ? cfg_nsl : nsl, q);
                if (rc != BZ_OK) return rc;
                if (!cfg_nsl && nsl > 1 && (q.l.grid > kGemmSlicedGrid || q.nsl != nsl)) continue;
                const float t = gemm_cost(wf, M, N, K, mt, nt, q);
                if (!found || t < best) {
                    best = t;
                    pl = q;
                    found = true;
                }
                if (cfg_nsl) break;
            }
        }
    return found ? BZ_OK : BZ_ERR_INVALID_ARG;
}

static int gemm_check(int wf, int M, int N, int K) {
    if (M < 1 || N < 1 || K < 1) return BZ_ERR_INVALID_ARG;
    if (wf != BZ_W_INT4_TILED && wf != BZ_W_FP8_TILED) return BZ_ERR_INVALID_ARG;
    if (N % 16 || !tiled_units(wf, K)) return BZ_ERR_SHAPE;
    return BZ_OK;
}

}  // namespace bz

using namespace bz;

extern "C" size_t bz_gemm_workspace(int32_t wfmt, int32_t M, int32_t N, int32_t K, int32_t cfg) {
    GemmPlan pl;
    if (gemm_check(wfmt, M, N, K) != BZ_OK || cfg < 0) return 0;
    return gemm_plan(wfmt, M, N, K, cfg & 255, (cfg >> 8) & 255, cfg >> 16, pl) == BZ_OK ? pl.ws : 0;
}

extern "C" int bz_gemm_tiled(int32_t wfmt, const void* x, int64_t ldx, int32_t M, const void* w, int32_t N, int32_t K,
                             void* out, int64_t ldo, int32_t out_dtype, void* workspace, size_t workspace_bytes,
                             int32_t cfg, void* stream) {
    if (!x || !w || !out || cfg < 0) return BZ_ERR_INVALID_ARG;
    if (out_dtype != BZ_DT_BF16 && out_dtype != BZ_DT_F32) return BZ_ERR_INVALID_ARG;
    const int rc = gemm_check(wfmt, M, N, K);
    if (rc != BZ_OK) return rc;
    if (ldx < K || ldo < N) return BZ_ERR_INVALID_ARG;
    auto off = [](const void* q, uintptr_t a) { return (reinterpret_cast<uintptr_t>(q) & (a - 1)) != 0; };
    if (off(x, 16) || ldx % 8 || off(w, 16) || off(out, out_dtype == BZ_DT_F32 ? 4 : 2)) return BZ_ERR_ALIGNMENT;
    if (ldx > (int64_t)1 << 22) return BZ_ERR_UNSUPPORTED;  // 32-bit offsets within a row tile
    GemmPlan pl;
    const int prc = gemm_plan(wfmt, M, N, K, cfg & 255, (cfg >> 8) & 255, cfg >> 16, pl);
    if (prc != BZ_OK) return prc;
    if (pl.ws && (!workspace || off(workspace, 16) || workspace_bytes < pl.ws)) return BZ_ERR_INVALID_ARG;
    GemmParams p{};
    p.x = static_cast<const uint16_t*>(x);
    p.ldx = ldx;
    p.w = static_cast<const uint8_t*>(w);
    p.NU = tiled_units(wfmt, K);
    p.chunk = tiled_chunk_bytes(wfmt, p.NU);
    p.out = out;
    p.ldo = ldo;
    p.part = static_cast<float*>(workspace);
    p.M = M;
    p.K = K;
    p.nblk = N / 16;
    p.mtiles = pl.mtiles;
    p.ntiles = pl.ntiles;
    p.nsl = pl.nsl;
    p.sps = pl.sps;
    p.out_f32 = out_dtype == BZ_DT_F32;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int lrc = wfmt == BZ_W_INT4_TILED ? launch_gemm_i4t(p, pl.l, st) : launch_gemm_f8t(p, pl.l, st);
    if (lrc != BZ_OK || pl.nsl == 1) return lrc;
    const int64_t items = (int64_t)M * (N / 4);
    hipLaunchKernelGGL(gemm_sum_slices, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, st, p.part, pl.nsl, M, N,
                       out, ldo, p.out_f32);
    return hipGetLastError() == hipSuccess ? BZ_OK : BZ_ERR_LAUNCH;
}
