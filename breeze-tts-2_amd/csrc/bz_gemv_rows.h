// Decode GEMV over plain bf16 weights [N][K]: the unquantized projections of
// a fused layer, for up to 4 rows of x per launch.
//
// Replaces rms_gemv_kernel + gemv_epilogue_kernel for bf16 weights
// (models/fused/kernels.py:41-138).
//
// Work decomposition
//   * A wave owns R weight rows over a span of 512 KC of K: lane l reads the
//     16 bytes at 8 l + 512 c of each row (1 KiB of a row per instruction),
//     and holds exactly the x values those meet, so x needs no LDS, no
//     barrier and no staging: it goes from L2 into the registers that
//     v_dot2_f32_bf16 reads.  All R KC weight loads of a wave are in flight at
//     once, behind its x loads.
//   * Rows longer than one span are split over KS = 2 or 4 waves of the
//     workgroup, whose sums meet in LDS (the only barrier).
//   * The wave's R M sums are reduced over its lanes by DPP, in a fixed order.
//   * Bound by HBM: 1.67 us of launch plus the bytes at the 7.39 TB/s of a plain
//     read is 3.94 us for N4096 K2048 and 2.81 for N2048 K2048; it takes 4.65
//     and 3.48 at M = 1, 5.01 and 3.65 at M = 2 (graph replays over 1 GiB of
//     weight copies on MI355X).  The kernel that staged x in LDS behind a
//     barrier and walked its tiles through a rolling pipeline took 6.01, 4.94,
//     6.94 and 5.36.
//   * RMSNorm is folded as in the other GEMVs: u = bf16(gamma x), and 1/rms of
//     the row multiplies the finished sums.  A wave that spans K has the whole
//     row of x in its lanes.
#pragma once

#include "bz_gemv_kernel.h"

namespace bz {

constexpr int kRowsWaves = 4;       // waves per workgroup
constexpr int kRowsMaxM = 4;        // rows of x per launch
constexpr int kRowsMaxKc = 5;       // 512-k pieces per wave
constexpr int kRowsMaxK = 4 * 512 * kRowsMaxKc;

// Sum over the wave's 64 lanes, in lane 63.
__device__ __forceinline__ float wave_sum_lane63(float v) { return rows4_sum_lane63(sum16_dpp(v)); }

template <int M, int KC, int R, bool PAIR>
__global__ void __launch_bounds__(kRowsWaves * 64) gemv_rows(const uint16_t* hx, const uint8_t* hw, const uint16_t* hgamma,
                                                             int hldx, int hK, int hn_out, int hks, int hM, int hnorm,
                                                             GemvParams p) {
    __shared__ float red[kRowsWaves][(R + 1) * M];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ks = wave & (hks - 1);
    constexpr int OC = PAIR ? R / 2 : R;  // output columns per wave
    const int c0 = ((int)blockIdx.x * (kRowsWaves / hks) + wave / hks) * OC;
    const int k0 = ks * (KC * 512) + lane * 8;

    // x, then gamma, then the weights; a piece past K, a row of x past the
    // call's and a column past the output read as zeros without a request
    const __amdgpu_buffer_rsrc_t xrs = buffer_rsrc(hx, (uint32_t)(((hM - 1) * hldx + hK) * 2));
    u32x4 xv[M][KC], gv[KC], wv[R][KC];
    uint32_t kb[KC];
#pragma unroll
    for (int c = 0; c < KC; ++c) kb[c] = k0 + c * 512 < hK ? (uint32_t)(k0 + c * 512) * 2u : kBufferOob;
#pragma unroll
    for (int c = 0; c < KC; ++c)
#pragma unroll
        for (int m = 0; m < M; ++m)
            xv[m][c] = buffer_ld16(xrs, m < hM && kb[c] != kBufferOob ? kb[c] + (uint32_t)(m * hldx) * 2u : kBufferOob);
    if (hnorm) {
        const __amdgpu_buffer_rsrc_t grs = buffer_rsrc(hgamma, (uint32_t)hK * 2u);
#pragma unroll
        for (int c = 0; c < KC; ++c) gv[c] = buffer_ld16(grs, kb[c]);
    }
    __builtin_amdgcn_sched_barrier(0);
    auto row_of = [&](int r) { return PAIR ? c0 + (r >> 1) + (r & 1) * hn_out : c0 + r; };
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const bool live = (PAIR ? c0 + (r >> 1) : c0 + r) < hn_out;
        const __amdgpu_buffer_rsrc_t wrs =
            buffer_rsrc(hw + (int64_t)(live ? row_of(r) : 0) * hK * 2, live ? (uint32_t)hK * 2u : 0u);
#pragma unroll
        for (int c = 0; c < KC; ++c) wv[r][c] = buffer_ld16_nt(wrs, kb[c]);
    }
    // output i = (row i / OC, column c0 + i % OC) belongs to lane i
    const int om = lane / OC, oc = c0 + lane % OC;
    const bool mine = lane < OC * M && om < hM && oc < hn_out;
    RawWord resv = {0u, 0u};
    if (p.epi == BZ_EPI_RESIDUAL && mine) resv = ld_elem(p.res, p.res_f32 ? 2 : 1, (int64_t)om * p.ldr + oc);
    __builtin_amdgcn_sched_barrier(0);

    float ss[M];
#pragma unroll
    for (int m = 0; m < M; ++m) ss[m] = 0.0f;
    if (hnorm) {
#pragma unroll
        for (int c = 0; c < KC; ++c)
#pragma unroll
            for (int m = 0; m < M; ++m)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t v = xv[m][c][q], g = gv[c][q];
                    ss[m] = dot2(v, v, ss[m]);
                    xv[m][c][q] = pack_bf16x2(bf16_lo(v) * bf16_lo(g), bf16_hi(v) * bf16_hi(g));
                }
    }
    float acc[R][M];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[r][m] = 0.0f;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < KC; ++c)
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int m = 0; m < M; ++m) acc[r][m] = dot2(wv[r][c][q], xv[m][c][q], acc[r][m]);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[r][m] = wave_sum_lane63(acc[r][m]);
    if (hnorm) {
#pragma unroll
        for (int m = 0; m < M; ++m) ss[m] = wave_sum_lane63(ss[m]);
    }

    // lane i < OC M takes its output's sums: from lane 63, or (KS > 1) from
    // the KS waves of the row group through LDS, added in wave order
    float a = 0.0f, b = 0.0f, s2 = 0.0f;
    if (hks == 1) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const float sq = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ss[m]), 63));
            if (m == om) s2 = sq;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float t =
                    __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, acc[r][m]), 63));
                const int o = m * OC + (PAIR ? r >> 1 : r);
                if (PAIR && (r & 1)) {
                    if (lane == o) b = t;
                } else if (lane == o) {
                    a = t;
                }
            }
        }
    } else {
        if (lane == 63) {
#pragma unroll
            for (int m = 0; m < M; ++m) {
#pragma unroll
                for (int r = 0; r < R; ++r) red[wave][r * M + m] = acc[r][m];
                red[wave][R * M + m] = ss[m];
            }
        }
        __syncthreads();
        if (ks != 0) return;
        if (mine) {
            const int r = lane % OC * (PAIR ? 2 : 1);
            for (int w = 0; w < hks; ++w) {
                a += red[wave + w][r * M + om];
                if (PAIR) b += red[wave + w][(r + 1) * M + om];
                s2 += red[wave + w][R * M + om];
            }
        }
    }
    if (!mine) return;
    const float inv = hnorm ? rsqrtf(s2 / (float)hK + p.eps) : 1.0f;
    a *= inv;
    if (PAIR) a = silu(a) * (b * inv);
    if (p.epi == BZ_EPI_RESIDUAL) a += p.res_f32 ? __uint_as_float(resv.w) : bf16_lo(resv.w >> resv.shift);
    const int64_t oi = (int64_t)om * p.ldo + oc;
    if (p.out_f32)
        static_cast<float*>(p.out)[oi] = a;
    else
        static_cast<uint16_t*>(p.out)[oi] = f32_to_bf16(a);
}

// ---- host side -----------------------------------------------------------------

struct RowsLaunch {
    int m, kc, r, ks;
    bool pair;
    unsigned grid;
};

template <int M, int KC, int R, bool PAIR>
int launch_rows_kernel(const GemvParams& p, const RowsLaunch& l, int rows, hipStream_t st) {
    hipLaunchKernelGGL((gemv_rows<M, KC, R, PAIR>), dim3(l.grid), dim3(kRowsWaves * 64), 0, st, p.x, p.w, p.gamma,
                       (int)p.ldx, p.K, p.n_out, l.ks, rows, p.norm, p);
    return hipGetLastError() == hipSuccess ? BZ_OK : BZ_ERR_LAUNCH;
}

template <int M, int KC>
int launch_rows_r(const GemvParams& p, const RowsLaunch& l, int rows, hipStream_t st) {
    if (l.pair) {
        if (l.r == 2) return launch_rows_kernel<M, KC, 2, true>(p, l, rows, st);
        if (l.r == 4) return launch_rows_kernel<M, KC, 4, true>(p, l, rows, st);
        return BZ_ERR_INVALID_ARG;
    }
    switch (l.r) {
        case 2: return launch_rows_kernel<M, KC, 2, false>(p, l, rows, st);
        case 4: return launch_rows_kernel<M, KC, 4, false>(p, l, rows, st);
        default: return BZ_ERR_INVALID_ARG;
    }
}

template <int M>
int launch_rows_kc(const GemvParams& p, const RowsLaunch& l, int rows, hipStream_t st) {
    switch (l.kc) {
        case 1: return launch_rows_r<M, 1>(p, l, rows, st);
        case 2: return launch_rows_r<M, 2>(p, l, rows, st);
        case 3: return launch_rows_r<M, 3>(p, l, rows, st);
        case 4: return launch_rows_r<M, 4>(p, l, rows, st);
        case 5: return launch_rows_r<M, 5>(p, l, rows, st);
        default: return BZ_ERR_INVALID_ARG;
    }
}

// `rows` <= 4 rows of x (bz_gemv_rows.hip).
int launch_rows(const GemvParams& p, const RowsLaunch& l, int rows, hipStream_t st);

}  // namespace bz
