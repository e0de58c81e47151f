// Decode GEMV over an unpaired fp8 tiled weight with few row blocks: a
// workgroup takes only 4, 8 or 16 rows of a 16-row block, so that a projection
// to a narrow hidden size (N = 1024: 64 blocks) still occupies every CU.
//
// Replaces rms_gemv_kernel + gemv_epilogue_kernel without the norm prologue
// (models/fused/kernels.py:41-138): the down and output projections.
//
// Work decomposition
//   * One wave instruction reads 4 rows x 64 bytes of 4 consecutive tiles: lane
//     l holds 16 codes of row (l / 4) % 4 of its group, unit l / 16, piece l % 4
//     (16 lanes read 256 contiguous bytes).  RL of them, 4 rows apart, share
//     the lane's x.
//   * The x a lane needs (16 values per unit and row of x) goes from L2 into
//     its registers; there is no LDS staging.  x first, then the weights, all
//     loads of a wave in flight at once.
//   * gfx950's exact e4m3 -> bf16 conversion, then v_dot2_f32_bf16; the lanes of
//     a row meet by DPP and lane-row swaps, the waves (split over K) in LDS
//     behind the only barrier.
//   * Bound by HBM latency at these sizes.  Measured on MI355X with a residual
//     (graph replays over >= 1 GiB of weight copies; floor = 1.67 us + bytes at
//     7.39 TB/s), the one- or several-block kernel -> this one: N1024 K8192
//     (floor 2.81) M = 1 4.98 -> 3.62 us, M = 2 5.13 -> 4.26; N1024 K1024
//     (1.81) 2.67 -> 2.38, 2.75 -> 2.61; N2048 K6144 (3.37) 5.10 -> 4.25, 4.75
//     -> 4.52; N2560 K10240 (5.22) M = 1 7.14 -> 6.73.
#pragma once

#include "bz_gemv_stream.h"

namespace bz {

constexpr int kSlabMaxNi = 3;  // groups of 4 units per wave (16 waves: K <= 12288)

struct SlabLaunch {
    int m, rl, ni, nw;
    unsigned grid;
};

// Sum over the four 16-lane rows of a wave, in every lane.
__device__ __forceinline__ float rows4_sum(float v) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    const float t = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(t), __float_as_uint(t), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

template <int M, int RL, int NI>
__global__ void __launch_bounds__(1024) gemv_slab(const uint8_t* hw, const uint16_t* hx, int hchunk, int hldx, int hK,
                                                  int hNU, int hM, StreamParams p) {
    __shared__ float red[4 * RL * M][16];  // [row][x row] by wave
    constexpr int RQ = 4 * RL, PB = 16 / RQ;  // rows per workgroup, workgroups per block
    const int tid = threadIdx.x, lane = tid & 63, NW = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int blk = (int)blockIdx.x / PB, r0 = ((int)blockIdx.x % PB) * RQ;
    const int u0 = wave * NI * 4 + (lane >> 4), rr = (lane >> 2) & 3, piece = lane & 3;
    const uint8_t* chunk = hw + (int64_t)blk * hchunk;

    const __amdgpu_buffer_rsrc_t xrs = buffer_rsrc(hx, (uint32_t)(((int64_t)(hM - 1) * hldx + hK) * 2));
    const __amdgpu_buffer_rsrc_t wrs = buffer_rsrc(chunk, (uint32_t)hNU * 1024u);
    u32x4 xv[NI][M][2], wv[NI][RL];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int u = u0 + 4 * i;
            const uint32_t o =
                u < hNU && m < hM ? (uint32_t)(((int64_t)m * hldx + u * 64 + piece * 16) * 2) : kBufferOob;
            xv[i][m][0] = buffer_ld16(xrs, o);
            xv[i][m][1] = buffer_ld16(xrs, o == kBufferOob ? o : o + 16);
        }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int t = 0; t < RL; ++t)
            wv[i][t] = buffer_ld16_nt(wrs, (uint32_t)(u0 + 4 * i) * 1024u + (r0 + 4 * t + rr) * 64 + piece * 16);
    __builtin_amdgcn_sched_barrier(0);
    // output g = (row, x row) belongs to the 16 lanes of group g: its row
    // scale and residual
    constexpr int kOut = RQ * M;
    const int g = min(tid >> 4, kOut - 1), gw = tid & 15;
    const int orow = r0 + g / M, om = g % M;
    const float rs = reinterpret_cast<const float*>(chunk + (int64_t)hNU * 1024)[orow];
    const int log2 = p.res_f32 ? 2 : 1;
    const int64_t ri = (int64_t)min(om, hM - 1) * p.ldr + blk * 16 + orow;
    RawWord resv = {0u, 0u};
    if (p.epi == BZ_EPI_RESIDUAL) resv = ld_elem(p.res, log2, ri);
    __builtin_amdgcn_sched_barrier(0);

    float acc[RL][M];
#pragma unroll
    for (int t = 0; t < RL; ++t)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[t][m] = 0.0f;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int t = 0; t < RL; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t lo = fp8x2_bf16<false>(wv[i][t][q]), hi = fp8x2_bf16<true>(wv[i][t][q]);
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    acc[t][m] = dot2(lo, xv[i][m][q >> 1][2 * (q & 1)], acc[t][m]);
                    acc[t][m] = dot2(hi, xv[i][m][q >> 1][2 * (q & 1) + 1], acc[t][m]);
                }
            }
#pragma unroll
    for (int t = 0; t < RL; ++t)
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const float v = rows4_sum(sum4(acc[t][m]));
            if (lane < 16 && piece == 0) red[(4 * t + rr) * M + m][wave] = v;
        }
    __syncthreads();
    if ((tid >> 4) >= kOut) return;
    const float a = sum16_dpp(gw < NW ? red[g][gw] : 0.0f);
    if (gw != 0 || om >= hM) return;
    float o = a * rs;
    if (p.epi == BZ_EPI_RESIDUAL) o += p.res_f32 ? __uint_as_float(resv.w) : bf16_lo(resv.w >> resv.shift);
    const int64_t oi = (int64_t)om * p.ldo + blk * 16 + orow;
    if (p.out_f32)
        static_cast<float*>(p.out)[oi] = o;
    else
        static_cast<uint16_t*>(p.out)[oi] = f32_to_bf16(o);
}

// ---- host side -----------------------------------------------------------------

template <int M, int RL, int NI>
int launch_slab_kernel(const StreamParams& p, const SlabLaunch& l, hipStream_t st) {
    if (!stream_hot_ok(p)) return BZ_ERR_UNSUPPORTED;
    hipLaunchKernelGGL((gemv_slab<M, RL, NI>), dim3(l.grid), dim3(l.nw * 64), 0, st, p.w, p.x, (int)p.chunk, (int)p.ldx,
                       p.K, p.NU, p.M, p);
    return hipGetLastError() == hipSuccess ? BZ_OK : BZ_ERR_LAUNCH;
}

// (the shapes the rule takes: 16 rows per workgroup for one row of x only;
// 3 and 4 rows of x over 4 rows and one group per wave)
template <int M, int RL>
int launch_slab_ni(const StreamParams& p, const SlabLaunch& l, hipStream_t st) {
    if (l.ni == 1) return launch_slab_kernel<M, RL, 1>(p, l, st);
    if constexpr (M <= 2) {
        switch (l.ni) {
            case 2: return launch_slab_kernel<M, RL, 2>(p, l, st);
            case 3: return launch_slab_kernel<M, RL, 3>(p, l, st);
            default: break;
        }
    }
    return BZ_ERR_INVALID_ARG;
}

template <int M>
int launch_slab_rl(const StreamParams& p, const SlabLaunch& l, hipStream_t st) {
    if (l.rl == 1) return launch_slab_ni<M, 1>(p, l, st);
    if constexpr (M <= 2)
        if (l.rl == 2) return launch_slab_ni<M, 2>(p, l, st);
    if constexpr (M == 1)
        if (l.rl == 4) return launch_slab_ni<M, 4>(p, l, st);
    return BZ_ERR_INVALID_ARG;
}

// bz_gemv_slab.hip
int launch_slab(const StreamParams& p, const SlabLaunch& l, hipStream_t st);

}  // namespace bz
