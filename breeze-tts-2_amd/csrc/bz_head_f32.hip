// fp32 output heads (gfx950): out[m][n] = sum_k x[m][k] * W[n][k], all fp32,
// for the per-frame heads the reference keeps unquantized and casts to fp32
// (backbone lm_head, models/cudagraph/backbone_graph.py:69-70,273; depth
// BreezeCodebooksHead, models/breeze.py:590-614 with
// models/cudagraph/depth_decoder_graph.py:159-161).
//
// W is one of `nmat` matrices [N][K] (K contiguous) spaced `mat_stride`
// floats apart; the matrix is w + sel * mat_stride with
// sel = *index + index_offset read on the device (index NULL: sel =
// index_offset), so a codebook chosen by a device cache position needs no
// host round trip and can sit in a captured graph.  A selection outside
// [0, nmat) writes zeros.
//
// Layout of the work: x rows (up to kHeadMaxRows per launch) in LDS as fp32,
// loaded into registers before the first weights are requested (vector loads
// retire in order, so staging x then waits for x alone); each wave owns
// kHeadRowsPerWave output rows n and streams them with 16-byte loads (64
// lanes cover 256 k per load), up to 8 such loads per row issued together
// so a 2048-k row takes one memory round trip; fp32 products are summed per
// lane in k order, then across the wave (DPP row sums, rows 0..3 in order).
//
// bz_norm_head_f32 also takes the decoder's final RMSNorm (bf16 x, gamma): the
// workgroup norms the rows of x while its weights are on their way, with the
// sums of rmsnorm_kernel (bz_aux.hip) and its rounding to bf16, so norm and
// head are one launch with the same results; and, for cond / uncond rows, the
// guidance combination of the logits it has just summed.  Measured on MI355X
// in graph replays, norm, cast and head launches -> this one: N2051 K1024 2
// rows 9.0 -> 4.7 us, 4 rows 11.1 -> 6.8; N2052 K2048 2 rows 12.6 -> 7.5 with the
// guidance.
#include "bz_device.h"
#include "bz_gemv.h"

namespace bz {

constexpr int kHeadThreads = 256;
constexpr int kHeadWaves = kHeadThreads / 64;
constexpr int kHeadRowsPerWave = 2;
constexpr int kHeadMaxRows = 4;                  // x rows per launch
constexpr int kHeadMaxK = 4096;
// the x rows in dynamic LDS, within the 64 KB that a launch may ask for without
// raising the kernel's limit (the fused form has 64 bytes of static sums beside)
static_assert(kHeadMaxRows * kHeadMaxK * sizeof(float) <= 65536, "dynamic LDS of the largest head");

__device__ __forceinline__ float head_row_sum(float v) {
    v += dpp_f32<kDppXor1>(v);
    v += dpp_f32<kDppXor2>(v);
    v += dpp_f32<0x124>(v);  // row_ror:4
    v += dpp_f32<0x128>(v);  // row_ror:8
    const int b = __float_as_int(v);
    return ((__int_as_float(__builtin_amdgcn_readlane(b, 0)) + __int_as_float(__builtin_amdgcn_readlane(b, 16))) +
            __int_as_float(__builtin_amdgcn_readlane(b, 32))) +
           __int_as_float(__builtin_amdgcn_readlane(b, 48));
}

// The fused form's inputs and outputs beside the head's.
struct HeadNorm {
    const uint16_t* x;      // bf16 rows, NULL: fp32 x without a norm
    const uint16_t* gamma;  // NULL: the bf16 rows as they are
    float eps;
    uint16_t* normed;       // optional: the normed rows, bf16
    int64_t ldn;
    float* cfg;             // optional: [M / 2] combined rows (or the row of M = 1)
    int64_t ldc;
    float guidance;
};

// S = 256-k loads per row issued together (min(8, K / 256), so no load is
// issued past a row for K a multiple of 256 S; the last chunk of other K
// clamps its indices into the row).  XN > 0: the fused form, K <= 256 XN; a
// thread loads XN elements of each row and of gamma whatever K is (N2052 K2560,
// 1, 2 and 4 bf16 rows: XN = 16 7.03, 8.87, 12.30 us, XN = 10 6.59, 8.32, 11.26;
// a cast launch and the fp32 form 8.39, 9.51, 12.18).
// EXACT: K = 256 S in one chunk, no guards (each was a branch that waited for
// the LDS reads before it) and no spare x loads: K = 1024 and 2048, the two
// heads' widths; other multiples of 256 run guarded.  Measured on MI355X (graph
// replays, 1, 2 and 4 rows): N2051 K1024 4.35, 5.06, 6.88 -> 3.67, 4.33, 5.35
// us; N2052 K2048 5.67, 6.56, 8.76 -> 5.29, 6.13, 7.59.
template <int M, int S, int XN, bool EXACT>
__global__ void __launch_bounds__(kHeadThreads) head_f32_kernel(const float* x, int64_t ldx, int argK, const float* w,
                                                               int64_t mat_stride, int nmat, const int64_t* index,
                                                               int64_t index_offset, int N, float* out, int64_t ldo,
                                                               HeadNorm hn) {
    extern __shared__ float xs[];  // [M][K]
    const int K = EXACT ? 256 * S : argK;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t sel = (index ? *index : 0) + index_offset;
    const bool ok = sel >= 0 && sel < nmat;
    const float* wm = w + (ok ? sel : 0) * mat_stride;
    const int n0 = (blockIdx.x * kHeadWaves + wave) * kHeadRowsPerWave;  // rows past N load row N - 1

    // 1. x into registers first (float4 e = tid + 256 i: row 4e / K), so
    //    waiting for it does not wait for the weights issued after it.  bf16
    //    rows to norm: element k = tid + 256 i of each row, and its gamma
    constexpr bool NORM = XN > 0;
    constexpr int XV = NORM ? 1 : M * (EXACT ? 256 * S : kHeadMaxK) / (4 * kHeadThreads);
    const int nx = M * (K >> 2);
    float4 xr[XV];
    uint16_t xb[NORM ? XN : 1][M], gb[NORM ? XN : 1];
    if constexpr (NORM) {
#pragma unroll
        for (int i = 0; i < XN; ++i) {
            const int k = min(tid + i * kHeadThreads, K - 1);
#pragma unroll
            for (int m = 0; m < M; ++m) xb[i][m] = hn.x[m * ldx + k];
            gb[i] = hn.gamma ? hn.gamma[k] : (uint16_t)0;
        }
        __builtin_amdgcn_sched_barrier(0);
    } else {
#pragma unroll
        for (int i = 0; i < XV; ++i) {
            const int e = min(tid + i * kHeadThreads, nx - 1);
            const int m = (4 * e) / K;
            xr[i] = *reinterpret_cast<const float4*>(x + m * ldx + (4 * e - m * K));
        }
    }
    // 2. the first chunk of weights (S loads of 256 k per row)
    const float* wrow[kHeadRowsPerWave];
    for (int r = 0; r < kHeadRowsPerWave; ++r) wrow[r] = wm + (int64_t)min(n0 + r, N - 1) * K;
    float4 wv[S][kHeadRowsPerWave];
    auto load_chunk = [&](int k0) {
#pragma unroll
        for (int u = 0; u < S; ++u) {
            const int k = min(k0 + 256 * u + 4 * lane, K - 4);
#pragma unroll
            for (int r = 0; r < kHeadRowsPerWave; ++r) wv[u][r] = *reinterpret_cast<const float4*>(wrow[r] + k);
        }
    };
    load_chunk(0);  // (no scheduling barrier here: one made the compiler spill xr)
    // 3. stage x (clamped entries hold element nx - 1 and store it again:
    //    unconditional stores keep xr in registers), or norm it first
    if constexpr (NORM) {
        __builtin_amdgcn_sched_barrier(0);
        __shared__ float part[M][kHeadWaves];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            float ss = 0.0f;
#pragma unroll
            for (int i = 0; i < XN; ++i) {
                const float v = bf16_to_f32(xb[i][m]);
                if (tid + i * kHeadThreads < K) ss += v * v;
            }
            ss = wave_sum(ss);
            if (lane == 0) part[m][wave] = ss;
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const bool plain = !hn.gamma;  // uniform
            const float inv = rsqrtf(((part[m][0] + part[m][1]) + (part[m][2] + part[m][3])) / (float)K + hn.eps);
#pragma unroll
            for (int i = 0; i < XN; ++i) {
                const int k = tid + i * kHeadThreads;
                if (k < K) {
                    const uint16_t o =
                        plain ? xb[i][m] : f32_to_bf16(bf16_to_f32(xb[i][m]) * inv * bf16_to_f32(gb[i]));
                    xs[m * K + k] = bf16_to_f32(o);
                    if (hn.normed && blockIdx.x == 0) hn.normed[m * hn.ldn + k] = o;
                }
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < XV; ++i) {
            const int e = min(tid + i * kHeadThreads, nx - 1);
            *reinterpret_cast<float4*>(xs + 4 * e) = xr[i];
        }
    }
    __syncthreads();
    if (n0 >= N) return;

    float acc[kHeadRowsPerWave][M];
    for (int r = 0; r < kHeadRowsPerWave; ++r)
        for (int m = 0; m < M; ++m) acc[r][m] = 0.0f;
    for (int k0 = 0; k0 < K; k0 += 256 * S) {
#pragma unroll
        for (int u = 0; u < S; ++u) {
            const int k = k0 + 256 * u + 4 * lane;
            if (EXACT || k < K) {  // lane-uniform except in a row's last chunk
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    const float4 xv = *reinterpret_cast<const float4*>(xs + m * K + k);
#pragma unroll
                    for (int r = 0; r < kHeadRowsPerWave; ++r)
                        acc[r][m] += wv[u][r].x * xv.x + wv[u][r].y * xv.y + wv[u][r].z * xv.z + wv[u][r].w * xv.w;
                }
            }
        }
        if (k0 + 256 * S < K) {
            load_chunk(k0 + 256 * S);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    for (int r = 0; r < kHeadRowsPerWave; ++r) {
        float s[M];
        for (int m = 0; m < M; ++m) {
            s[m] = head_row_sum(acc[r][m]);
            if (!ok) s[m] = 0.0f;
            if (lane == 0 && n0 + r < N) out[m * ldo + n0 + r] = s[m];
        }
        if constexpr (NORM) {
            if (hn.cfg && lane == 0 && n0 + r < N) {
                constexpr int H = M == 1 ? 1 : M / 2;
                for (int h = 0; h < H; ++h)
                    hn.cfg[h * hn.ldc + n0 + r] = M == 1 ? s[0] : s[H + h] + hn.guidance * (s[h] - s[H + h]);
            }
        }
    }
}

struct HeadCall {
    const float* x;
    int64_t ldx;
    int K;
    const float* w;
    int64_t mat_stride;
    int nmat;
    const int64_t* index;
    int64_t index_offset;
    int N;
    float* out;
    int64_t ldo;
    HeadNorm hn;
};

template <int M, int S, int XN, bool EXACT>
static void launch_head_s(const HeadCall& c, hipStream_t st) {
    const int per_block = kHeadWaves * kHeadRowsPerWave;
    hipLaunchKernelGGL((head_f32_kernel<M, S, XN, EXACT>), dim3((c.N + per_block - 1) / per_block), dim3(kHeadThreads),
                       (size_t)M * c.K * sizeof(float), st, c.x, c.ldx, c.K, c.w, c.mat_stride, c.nmat, c.index,
                       c.index_offset, c.N, c.out, c.ldo, c.hn);
}

template <int M, bool NORM>
static void launch_head_m(const HeadCall& c, hipStream_t st) {
    // without a norm a chunk's loads never run past a row; the normed rows
    // need K <= 256 XN
    constexpr int X4 = NORM ? 4 : 0, X8 = NORM ? 8 : 0;
    if (c.K == 2048)
        launch_head_s<M, 8, X8, true>(c, st);
    else if (c.K == 1024)
        launch_head_s<M, 4, X4, true>(c, st);
    else if (NORM && c.K > 2048 && c.K <= 2560)
        launch_head_s<M, 8, NORM ? 10 : 0, false>(c, st);
    else if (NORM ? c.K > 2048 : c.K >= 2048)
        launch_head_s<M, 8, NORM ? 16 : 0, false>(c, st);
    else if (NORM && c.K > 1024)
        launch_head_s<M, 8, X8, false>(c, st);
    else if (NORM || c.K >= 1024)
        launch_head_s<M, 4, X4, false>(c, st);
    else if constexpr (!NORM) {
        if (c.K >= 512)
            launch_head_s<M, 2, 0, false>(c, st);
        else
            launch_head_s<M, 1, 0, false>(c, st);
    }
}

template <bool NORM>
static void launch_head(int rows, const HeadCall& c, hipStream_t st) {
    switch (rows) {
        case 1: launch_head_m<1, NORM>(c, st); break;
        case 2: launch_head_m<2, NORM>(c, st); break;
        case 3: launch_head_m<3, NORM>(c, st); break;
        default: launch_head_m<4, NORM>(c, st); break;
    }
}

static int check_head(int32_t M, int32_t K, const float* w, int32_t N, int64_t mat_stride, int32_t nmat, const void* x,
                      int64_t ldx, const float* out, int64_t ldo) {
    if (!x || !w || !out) return BZ_ERR_INVALID_ARG;
    if (M < 1 || N < 1 || K < 1 || nmat < 1 || mat_stride < 0) return BZ_ERR_INVALID_ARG;
    if (nmat > 1 && mat_stride < (int64_t)N * K) return BZ_ERR_SHAPE;
    if (K % 4 || K > kHeadMaxK || ldx < K || ldo < N || mat_stride % 4) return BZ_ERR_SHAPE;
    return reinterpret_cast<uintptr_t>(w) & 15 ? BZ_ERR_ALIGNMENT : BZ_OK;
}

}  // namespace bz

using namespace bz;

extern "C" int bz_head_f32(const float* x, int64_t ldx, int32_t M, int32_t K, const float* w, int32_t N,
                           int64_t mat_stride, int32_t nmat, const int64_t* index, int64_t index_offset, float* out,
                           int64_t ldo, void* stream) {
    const int rc = check_head(M, K, w, N, mat_stride, nmat, x, ldx, out, ldo);
    if (rc != BZ_OK && rc != BZ_ERR_ALIGNMENT) return rc;
    if (ldx % 4) return BZ_ERR_SHAPE;
    if (rc != BZ_OK || (reinterpret_cast<uintptr_t>(x) & 15)) return BZ_ERR_ALIGNMENT;
    HeadCall c{x, ldx, K, w, mat_stride, nmat, index, index_offset, N, out, ldo, HeadNorm{}};
    for (int m0 = 0; m0 < M; m0 += kHeadMaxRows) {
        c.x = x + (int64_t)m0 * ldx;
        c.out = out + (int64_t)m0 * ldo;
        launch_head<false>(M - m0 < kHeadMaxRows ? M - m0 : kHeadMaxRows, c, static_cast<hipStream_t>(stream));
        if (hipGetLastError() != hipSuccess) return BZ_ERR_LAUNCH;
    }
    return BZ_OK;
}

extern "C" int bz_norm_head_f32(const void* x, int64_t ldx, int32_t M, int32_t K, const void* gamma, float eps,
                                void* normed, int64_t ld_normed, const float* w, int32_t N, int64_t mat_stride,
                                int32_t nmat, const int64_t* index, int64_t index_offset, float* out, int64_t ldo,
                                float* cfg, int64_t ld_cfg, float guidance, void* stream) {
    const int rc = check_head(M, K, w, N, mat_stride, nmat, x, ldx, out, ldo);
    if (rc != BZ_OK) return rc;
    if (cfg && M > 1 && M % 2) return BZ_ERR_INVALID_ARG;
    if (M > kHeadMaxRows || (normed && ld_normed < K) || (cfg && ld_cfg < N)) return BZ_ERR_SHAPE;
    const HeadNorm hn{static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(gamma), eps,
                      static_cast<uint16_t*>(normed), ld_normed, cfg, ld_cfg, guidance};
    launch_head<true>(M, HeadCall{nullptr, ldx, K, w, mat_stride, nmat, index, index_offset, N, out, ldo, hn},
                      static_cast<hipStream_t>(stream));
    return hipGetLastError() == hipSuccess ? BZ_OK : BZ_ERR_LAUNCH;
}
