// Prefill GEMM over the unpaired tiled weight formats: out[M, N] = x[M, K] @
// w_eff[N, K]^T for the row counts of a prompt (33 and more), the weight
// decoded in registers on its way into the matrix cores.
//
// Stands where the reference runs, for M > 32 rows of a prompt,
//   torch._weight_int4pack_mm (Int4Linear)          models/int4_linear.py:103-108
//   torch._scaled_mm (Fp8Linear, weight-only form)  models/fp8_linear.py:76-82
//
// Bound by the matrix cores for long prompts and by the chain of loads, LDS
// and barrier of each step for short ones.  Measured on MI355X (graph replays,
// four weight copies in turn): int4 K2560 N10240 M = 203 23.5 us, int4 K10240
// N2560 M = 2048 116 us (926 TFLOP/s; a large bf16 matmul of the library
// reaches 1187 on the card), fp8 K2048 N6144 M = 1024 35.8 us (720), fp8
// K10240 N2560 M = 2048 98 us (1098).  Decoding the weight to fp32 in memory,
// casting it and running the library GEMM on the copy, in runs of 16 MB, took
// 286, 373, 129 and 320 us for the same calls.
//
// Work decomposition
//   * A workgroup of eight waves owns MT x 16 rows of x and 4 NT row blocks of
//     the weight and takes 256 k per step: wave (c, g) multiplies all of those
//     rows with its own NT blocks over half g of the step, so every weight
//     tile is loaded and decoded by exactly one wave of the workgroup,
//     straight from memory into registers: the tile's lane placement (lane
//     n + 16 g holds 16 bytes of row n) is the MFMA operand's.  The two K
//     halves give each SIMD a second wave over the same x (four waves over 128
//     k: 33.0, 168, 42.3 and 120 us for the calls above); they are added
//     through LDS at the end, each group finishing half of the rows.
//   * x goes through LDS, two buffers and one barrier per step.  A row of a
//     step is 2 x 16 pieces of 16 bytes; piece p of a half and row r sits at
//     p ^ (r % 16), so the 16 rows that one operand read touches lie on
//     different banks.  The pieces of a later step (one ahead, two where the
//     registers allow) are in flight in registers and written to the other
//     buffer at the end of a step.  Reading x costs MT LDS reads per MT NT
//     MFMAs: at NT = 3 the LDS is busy 5/6 of the MFMA time.
//   * Weights run two steps ahead in two register sets; operand d + 1 of a
//     unit is decoded while operand d is multiplied.
//   * Consecutive workgroups of one XCD (the dispatcher deals them out round
//     robin over 8) take neighbouring column tiles of one row tile, so they
//     read the same x from that XCD's L2.
//   * K slices (nsl > 1) for grids that would leave most of the chip idle:
//     each slice stores fp32 sums to the workspace [nsl][M][N] and a second
//     launch adds them in slice order.
//
// Arithmetic: v_mfma_f32_16x16x32_bf16, A = 16 weight rows, B = 16 rows of x;
// D[n][m] lands in lane m + 16 (n / 4), element n % 4, so a lane finishes four
// consecutive columns of one output row.
//   * int4: w = bf16((q - 8) s + z), the effective weight rounded to bf16 as
//     bz_dequant's float would be.  The lane's dword d holds k = 32 g + 8 d + 0..7:
//     one MFMA operand, met by piece 4 g + d of the x row's half.
//   * fp8: the exact bf16 value of each code; the row scale multiplies the
//     finished sum.  Codes 8 e..8 e+7 of lane row g in tile h of the half meet
//     piece 8 h + 2 g + e.
#pragma once

#include <type_traits>

#include "bz_gemv_stream.h"

namespace bz {

struct GemmParams {
    const uint16_t* x;
    int64_t ldx;
    const uint8_t* w;
    int64_t chunk;  // bytes per row block
    void* out;
    int64_t ldo;
    float* part;    // nsl > 1: fp32 sums [nsl][M][nblk * 16]
    int M, K, NU, nblk;
    int mtiles, ntiles, nsl, sps;  // tiles, K slices and steps per slice
    int out_f32;
};

constexpr int kGemmColWaves = 4;         // waves side by side over the columns
constexpr int kGemmKGroups = 2;          // and over the two units of a step
constexpr int kGemmThreads = kGemmColWaves * kGemmKGroups * 64;
constexpr int kGemmStepK = 256;
constexpr int kGemmMt[] = {2, 4, 6, 8};  // 16-row groups of x per workgroup
constexpr int kGemmNt[] = {1, 2, 3, 4};  // row blocks of the weight per wave

// accumulators of more tiles than these do not fit two waves per SIMD
__host__ __device__ constexpr bool gemm_shape_ok(int mt, int nt) { return mt * nt <= 24; }
__host__ __device__ constexpr int gemm_lds(int mt) { return 2 * mt * 16 * kGemmStepK * 2; }

// One dword of nibbles (k = 0..7) -> the four bf16 pairs of its effective
// weights: each nibble's float by the byte conversion, one fma, one rounding.
__device__ __forceinline__ u32x4 int4_weights(uint32_t v, float s, float zp) {
    uint32_t even = v & 0x0F0F0F0Fu, odd = (v >> 4) & 0x0F0F0F0Fu;
    // opaque: the known zero bits would turn each byte conversion
    // (v_cvt_f32_ubyte0..3) into a bit-field extract and a conversion
    asm("" : "+v"(even), "+v"(odd));
    u32x4 r;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const float q0 = (float)((even >> (8 * b)) & 0xFFu), q1 = (float)((odd >> (8 * b)) & 0xFFu);
        r[b] = pack_bf16x2(fmaf(q0, s, zp), fmaf(q1, s, zp));
    }
    return r;
}

template <int WF, int MT, int NT>
__global__ void __launch_bounds__(kGemmThreads, 2) gemm_tiled(GemmParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    constexpr bool I4 = tiled_i4(WF);
    constexpr int TPU = I4 ? 1 : 2;                // tiles per block and 128 k
    constexpr int PX = MT <= 4 || MT * NT <= 12 ? 2 : 1, PW = 2;  // steps ahead: x, weights
    constexpr int kBuf = MT * 16 * kGemmStepK * 2;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cw = wave & (kGemmColWaves - 1), kg = wave / kGemmColWaves;
    const int j = lane & 15, kq = lane >> 4;

    // this workgroup's tile: XCD c = bid % 8 takes a run of consecutive ids
    const int nwg = (int)gridDim.x, bid = (int)blockIdx.x;
    const int per = nwg >> 3, rem = nwg & 7, xcd = bid & 7;
    const int id = xcd * per + min(xcd, rem) + (bid >> 3);
    const int nt_i = id % p.ntiles, rest = id / p.ntiles;
    const int mt_i = rest % p.mtiles, sl = rest / p.mtiles;
    const int m0 = mt_i * MT * 16;
    const int steps = (p.K + kGemmStepK - 1) / kGemmStepK;
    const int s_begin = sl * p.sps, s_end = min(steps, s_begin + p.sps);
    const int blk0 = (nt_i * kGemmColWaves + cw) * NT;

    // x: thread t loads piece t % 32 of rows t / 32 + 16 i.  Rows past M and
    // pieces past K are out of the range (zeros, no request); the host keeps a
    // tile's range below kXOut.
    constexpr uint32_t kXOut = 0x80000000u;
    const int rows = min(p.M - m0, MT * 16);
    const __amdgpu_buffer_rsrc_t xrs =
        buffer_rsrc(p.x + (int64_t)m0 * p.ldx, (uint32_t)(((int64_t)(rows - 1) * p.ldx + p.K) * 2));
    const int xp = tid & 31, xr = tid >> 5;
    const uint32_t xo = (uint32_t)(xr * (int)p.ldx + xp * 8) * 2u, xstep = (uint32_t)p.ldx * 32u;
    const int xw = xr * 512 + (((xp & 16) | ((xp ^ xr) & 15)) << 4);
    u32x4 xv[PX][MT];
    auto x_load = [&](int set, int s) {
        const uint32_t o = s < s_end && s * kGemmStepK + xp * 8 < p.K ? xo + (uint32_t)s * (kGemmStepK * 2) : kXOut;
#pragma unroll
        for (int i = 0; i < MT; ++i) xv[set][i] = buffer_ld16(xrs, o + (uint32_t)i * xstep);
    };
    auto x_store = [&](int set, int buf) {
#pragma unroll
        for (int i = 0; i < MT; ++i) *reinterpret_cast<u32x4*>(smem + buf * kBuf + xw + i * 8192) = xv[set][i];
    };

    // weights and int4 scale pairs of the wave's blocks; a block past the
    // weight has an empty range, and the slice's tiles end at ue
    __amdgpu_buffer_rsrc_t wrs[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const bool live = blk0 + t < p.nblk;
        const uint8_t* c = p.w + (int64_t)(live ? blk0 + t : 0) * p.chunk;
        wrs[t] = buffer_rsrc(c, live ? (uint32_t)p.NU * (I4 ? 1088u : 1024u) : 0u);
    }
    const int ue = min(p.NU, s_end * kGemmKGroups * TPU);
    const uint32_t wl = j * 64 + kq * 16;
    u32x4 wv[PW][NT][TPU];
    uint32_t sz[PW][NT];
    auto w_load = [&](int set, int s) {
        const int u0 = (s * kGemmKGroups + kg) * TPU;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int h = 0; h < TPU; ++h)
                wv[set][t][h] = buffer_ld16(wrs[t], u0 + h < ue ? (uint32_t)(u0 + h) * 1024u + wl : kBufferOob);
            if (I4)
                sz[set][t] =
                    buffer_ld4(wrs[t], u0 < ue ? (uint32_t)p.NU * 1024u + (uint32_t)u0 * 64u + j * 4 : kBufferOob);
        }
    };
    // operand d (32 k) of the wave's unit
    auto decode = [&](u32x4 (&o)[NT], int set, int d) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if (I4) {
                const float sc = bf16_lo(sz[set][t]);
                o[t] = int4_weights(wv[set][t][0][d], sc, fmaf(-8.0f, sc, bf16_hi(sz[set][t])));
            } else {
                const u32x4 v = wv[set][t][TPU == 1 ? 0 : d >> 1];
                const uint32_t a = v[2 * (d & 1)], b = v[2 * (d & 1) + 1];
                o[t] = u32x4{fp8x2_bf16<false>(a), fp8x2_bf16<true>(a), fp8x2_bf16<false>(b), fp8x2_bf16<true>(b)};
            }
        }
    };

    f32x4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    // one step of 256 k: operand d of all rows and blocks while operand d + 1
    // is decoded
    auto step = [&](int set, int s, int buf) {
        const uint8_t* xb = smem + buf * kBuf + j * 512 + kg * 256;
        u32x4 wd[2][NT];
        decode(wd[0], set, 0);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const int piece = I4 ? 4 * kq + d : 8 * (d >> 1) + 2 * kq + (d & 1);
            if (d < 3) decode(wd[(d + 1) & 1], set, d + 1);
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const u32x4 xf = *reinterpret_cast<const u32x4*>(xb + i * 8192 + ((piece ^ j) << 4));
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[i][t] = mfma_bf16(wd[d & 1][t], xf, acc[i][t]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        w_load(set, s + PW);
        __builtin_amdgcn_sched_barrier(0);
        const int xs = PX == 2 ? buf ^ 1 : 0;
        x_store(xs, buf ^ 1);
        x_load(xs, s + 1 + PX);
        __syncthreads();
    };

    // the loads in the order the loop issues them (exact wait counts), then
    // whole pairs of steps: a step past the slice multiplies zeros
    x_load(0, s_begin);
    __builtin_amdgcn_sched_barrier(0);
    w_load(0, s_begin);
    __builtin_amdgcn_sched_barrier(0);
    if (PX == 2) x_load(1, s_begin + 1);
    __builtin_amdgcn_sched_barrier(0);
    w_load(1, s_begin + 1);
    __builtin_amdgcn_sched_barrier(0);
    x_store(0, 0);
    x_load(0, s_begin + PX);
    __syncthreads();
    int s = s_begin;
    do {
        step(0, s, 0);
        step(1, s + 1, 1);
        s += 2;
    } while (s < s_end);

    // the two K groups swap halves of their sums through LDS: group g finishes
    // the row groups of its parity
    f32x4_t* red = reinterpret_cast<f32x4_t*>(smem) + cw * MT * NT * 64 + lane;
    auto swap = [&](auto par) {
        constexpr int P = decltype(par)::value;
#pragma unroll
        for (int i = P ^ 1; i < MT; i += 2)
#pragma unroll
            for (int t = 0; t < NT; ++t) red[(i * NT + t) * 64] = acc[i][t];
        __syncthreads();
#pragma unroll
        for (int i = P; i < MT; i += 2)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[i][t] += red[(i * NT + t) * 64];
        // four consecutive columns of one row per lane and block
        const int n_out = p.nblk * 16;
        auto finish = [&](auto&& store) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if (blk0 + t >= p.nblk) continue;
                f32x4_t sc = {1.0f, 1.0f, 1.0f, 1.0f};
                if (!I4)
                    sc = *reinterpret_cast<const f32x4_t*>(p.w + (int64_t)(blk0 + t) * p.chunk + (int64_t)p.NU * 1024 +
                                                           kq * 16);
#pragma unroll
                for (int i = P; i < MT; i += 2) {
                    const int m = m0 + i * 16 + j;
                    if (m < p.M) store(m, (blk0 + t) * 16 + 4 * kq, I4 ? acc[i][t] : acc[i][t] * sc);
                }
            }
        };
        if (p.nsl > 1)
            finish([&](int m, int c, f32x4_t v) {
                *reinterpret_cast<f32x4_t*>(p.part + ((int64_t)sl * p.M + m) * n_out + c) = v;
            });
        else if (p.out_f32)
            finish([&](int m, int c, f32x4_t v) {
                float* o = static_cast<float*>(p.out) + (int64_t)m * p.ldo + c;
#pragma unroll
                for (int q = 0; q < 4; ++q) o[q] = v[q];
            });
        else
            finish([&](int m, int c, f32x4_t v) {
                uint16_t* o = static_cast<uint16_t*>(p.out) + (int64_t)m * p.ldo + c;
#pragma unroll
                for (int q = 0; q < 4; ++q) o[q] = f32_to_bf16(v[q]);
            });
    };
    if (kg == 0)
        swap(std::integral_constant<int, 0>{});
    else
        swap(std::integral_constant<int, 1>{});
}

struct GemmLaunch {
    int mt, nt;
    unsigned grid;
};

template <int WF, int MT, int NT>
int launch_gemm_kernel(const GemmParams& p, const GemmLaunch& l, hipStream_t st) {
    if constexpr (gemm_shape_ok(MT, NT)) {
        auto kern = gemm_tiled<WF, MT, NT>;
        constexpr int lds = gemm_lds(MT);
        if (lds > 65536 && raise_lds_limit(reinterpret_cast<const void*>(kern)) != BZ_OK) return BZ_ERR_LAUNCH;
        hipLaunchKernelGGL(kern, dim3(l.grid), dim3(kGemmThreads), lds, st, p);
        return hipGetLastError() == hipSuccess ? BZ_OK : BZ_ERR_LAUNCH;
    } else {
        return BZ_ERR_INVALID_ARG;
    }
}

template <int WF, int MT>
int launch_gemm_nt(const GemmParams& p, const GemmLaunch& l, hipStream_t st) {
    switch (l.nt) {
        case 1: return launch_gemm_kernel<WF, MT, 1>(p, l, st);
        case 2: return launch_gemm_kernel<WF, MT, 2>(p, l, st);
        case 3: return launch_gemm_kernel<WF, MT, 3>(p, l, st);
        case 4: return launch_gemm_kernel<WF, MT, 4>(p, l, st);
        default: return BZ_ERR_INVALID_ARG;
    }
}

template <int WF>
int launch_gemm_wf(const GemmParams& p, const GemmLaunch& l, hipStream_t st) {
    switch (l.mt) {
        case 2: return launch_gemm_nt<WF, 2>(p, l, st);
        case 4: return launch_gemm_nt<WF, 4>(p, l, st);
        case 6: return launch_gemm_nt<WF, 6>(p, l, st);
        case 8: return launch_gemm_nt<WF, 8>(p, l, st);
        default: return BZ_ERR_INVALID_ARG;
    }
}

// One instantiation set per unpaired tiled format (bz_gemm_<fmt>.hip).
int launch_gemm_i4t(const GemmParams& p, const GemmLaunch& l, hipStream_t st);
int launch_gemm_f8t(const GemmParams& p, const GemmLaunch& l, hipStream_t st);

}  // namespace bz
