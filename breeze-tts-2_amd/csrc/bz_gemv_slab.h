// Decode GEMV over an unpaired fp8 tiled weight with few row blocks: a
// workgroup takes only 4 rows of a 16-row block, so that a projection to a
// narrow hidden size (N = 1024: 64 blocks) still occupies every CU.
//
// Replaces rms_gemv_kernel + gemv_epilogue_kernel without the norm prologue
// (models/fused/kernels.py:41-138): the down and output projections.
//
// Work decomposition
//   * The K split is that of the one- or several-block kernel it stands in for
//     (NV waves of UPW consecutive units, one accumulator chain each, their
//     sums met in the same order), and so are the MFMAs a chain consists of:
//     the result is the same, bit for bit.  A token picked from it does not
//     depend on which kernel ran.
//   * v_mfma_f32_16x16x32_bf16 has room for 16 columns and 16 rows of x, the 4
//     weight rows and up to 4 rows of x need a quarter of each.  So one wave
//     runs the chains of 4 split-K parts side by side: column 4 c + row holds
//     the weight rows' codes of part c, row 4 m + c of A the x row m over part
//     c's units, and the products of unlike parts are dropped.  Each lane then
//     loads 16 bytes of weights per unit, 256 contiguous bytes per part.
//   * x goes from L2 into the registers of the A operand: no LDS staging.  x
//     first, then the weights, all loads of a wave in flight at once; the one
//     barrier is before the epilogue.
//   * Bound by HBM latency at these sizes.  Measured on MI355X with a residual
//     (graph replays over 1 GiB of weight copies; floor = 1.67 us + bytes at
//     7.39 TB/s), the kernel it stands in for -> this one, M = 1, 2, 4: N1024
//     K8192 (floor 2.81) 4.99 -> 3.92, 5.10 -> 4.01, 5.40 -> 4.42; N1024 K1024
//     (1.81) 2.66 -> 2.44, 2.75 -> 2.46, 3.00 -> 3.00; N2048 K2048 (2.24) 3.29 ->
//     3.06, 3.44 -> 3.13; N2048 K6144 (3.37) 5.05 -> 4.76, 4.73 -> 4.63.
#pragma once

#include "bz_gemv_stream.h"

namespace bz {

constexpr int kSlabRows = 4;      // weight rows per workgroup = split-K parts per wave
constexpr int kSlabMaxM = 4;      // rows of x
constexpr int kSlabMaxBlocks = 128;

struct SlabLaunch {
    int nv, upw;  // split-K parts and units per part, of the plan it stands in for
    int chain;    // 1: that plan adds its parts one after the other, 0: by a tree
    unsigned threads, grid;
};

template <int UPW>
__global__ void __launch_bounds__(256) gemv_slab(const uint8_t* hw, const uint16_t* hx, int hchunk, int hldx, int hNU,
                                                 int hM, int hnv, int hchain, StreamParams p) {
    __shared__ __attribute__((aligned(16))) float red[kSlabMaxM * kSlabRows][16];  // [x row, weight row][part]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int blk = (int)blockIdx.x >> 2, r0 = ((int)blockIdx.x & 3) * kSlabRows;
    const int j = lane & 15, kq = lane >> 4;
    const uint8_t* chunk = hw + (int64_t)blk * hchunk;
    // column j of B: weight row j % 4 over the units of part j / 4; row j of
    // A: x row j / 4 over the units of part j % 4
    const int ub = (wave * 4 + (j >> 2)) * UPW, ua = (wave * 4 + (j & 3)) * UPW, xm = j >> 2;

    const __amdgpu_buffer_rsrc_t xrs =
        buffer_rsrc(hx, (uint32_t)(((int64_t)(hM - 1) * hldx + (int64_t)hNU * 64) * 2));
    const __amdgpu_buffer_rsrc_t wrs = buffer_rsrc(chunk, (uint32_t)hNU * 1024u);
    // a unit past the row and a row of x past the call's read as zeros without
    // a request, and add 0
    u32x4 xv[UPW][2], wv[UPW];
#pragma unroll
    for (int q = 0; q < UPW; ++q) {
        const uint32_t o = xm < hM && ua + q < hNU
                               ? (uint32_t)(((int64_t)xm * hldx + (ua + q) * 64 + kq * 16) * 2)
                               : kBufferOob;
        xv[q][0] = buffer_ld16(xrs, o);
        xv[q][1] = buffer_ld16(xrs, o == kBufferOob ? o : o + 16);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < UPW; ++q)
        wv[q] = buffer_ld16_nt(wrs, (uint32_t)(ub + q) * 1024u + (r0 + (j & 3)) * 64 + kq * 16);
    __builtin_amdgcn_sched_barrier(0);
    // output g = (x row, weight row) belongs to the 16 lanes of group g: its
    // row scale and residual
    const int g = min(tid >> 4, hM * kSlabRows - 1), gw = tid & 15;
    const int om = g / kSlabRows, orow = r0 + g % kSlabRows;
    const float rs = reinterpret_cast<const float*>(chunk + (int64_t)hNU * 1024)[orow];
    RawWord resv = {0u, 0u};
    if (p.epi == BZ_EPI_RESIDUAL) resv = ld_elem(p.res, p.res_f32 ? 2 : 1, (int64_t)om * p.ldr + blk * 16 + orow);
    __builtin_amdgcn_sched_barrier(0);

    f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int q = 0; q < UPW; ++q) {
        const u32x4 b0 = {fp8x2_bf16<false>(wv[q][0]), fp8x2_bf16<true>(wv[q][0]), fp8x2_bf16<false>(wv[q][1]),
                          fp8x2_bf16<true>(wv[q][1])};
        const u32x4 b1 = {fp8x2_bf16<false>(wv[q][2]), fp8x2_bf16<true>(wv[q][2]), fp8x2_bf16<false>(wv[q][3]),
                          fp8x2_bf16<true>(wv[q][3])};
        acc = mfma_bf16(xv[q][0], b0, acc);
        acc = mfma_bf16(xv[q][1], b1, acc);
    }
    // lane (j, kq) holds rows 4 kq + e of column j: x row kq, its own part at e = j / 4
    const int part = j >> 2;
    const float y = part == 0 ? acc[0] : part == 1 ? acc[1] : part == 2 ? acc[2] : acc[3];
    red[kq * kSlabRows + (j & 3)][(wave * 4 + part) & 15] = y;
    __syncthreads();
    if ((tid >> 4) >= hM * kSlabRows) return;
    float a = 0.0f;
    if (hchain) {  // in order, as the several-block kernel adds its waves
#pragma unroll
        for (int w = 0; w < 16; w += 4) {
            const float4 v = *reinterpret_cast<const float4*>(&red[g][w]);
            a = (((a + (w < hnv ? v.x : 0.0f)) + (w + 1 < hnv ? v.y : 0.0f)) + (w + 2 < hnv ? v.z : 0.0f)) +
                (w + 3 < hnv ? v.w : 0.0f);
        }
    } else {
        a = sum16_dpp(gw < hnv ? red[g][gw] : 0.0f);
    }
    if (gw != 0) return;
    float o = a * rs;
    if (p.epi == BZ_EPI_RESIDUAL) o += p.res_f32 ? __uint_as_float(resv.w) : bf16_lo(resv.w >> resv.shift);
    const int64_t oi = (int64_t)om * p.ldo + blk * 16 + orow;
    if (p.out_f32)
        static_cast<float*>(p.out)[oi] = o;
    else
        static_cast<uint16_t*>(p.out)[oi] = f32_to_bf16(o);
}

// ---- host side -----------------------------------------------------------------

template <int UPW>
int launch_slab_kernel(const StreamParams& p, const SlabLaunch& l, hipStream_t st) {
    if (!stream_hot_ok(p)) return BZ_ERR_UNSUPPORTED;
    hipLaunchKernelGGL((gemv_slab<UPW>), dim3(l.grid), dim3(l.threads), 0, st, p.w, p.x, (int)p.chunk, (int)p.ldx, p.NU,
                       p.M, l.nv, l.chain, p);
    return hipGetLastError() == hipSuccess ? BZ_OK : BZ_ERR_LAUNCH;
}

// bz_gemv_slab.hip
int launch_slab(const StreamParams& p, const SlabLaunch& l, hipStream_t st);

}  // namespace bz
