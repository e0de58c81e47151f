// Decode-step attention of the fused decoder layer (gfx950): one new token
// per batch row against a static KV cache.
//
// Reference behaviour replaced (models/fused/kernels.py):
//   _rms_head, _rope, qkv_rope_cache_kernel :356-401  per-head q/k RMSNorm,
//       rotate-half RoPE, q to fp32, new k and v into the cache at pos
//   attn_decode_kernel                       :404-453  softmax(q k^T scale +
//       mask) v over the cache positions [0, pos], split over positions
//   attn_combine_kernel, attention_step      :456-536
//
// Layouts: qkv bf16 [B][ld_qkv] = [q heads | k heads | v heads] x D; caches
// [B][HKV][S][D] (bf16 or fp32); cos/sin [B or 1][D] (bf16 or fp32, batch
// stride ld_cs, 0 to broadcast one row); mask [B][ld_mask] additive bf16 or
// fp32, or bool (ld_mask 0: one row for all);
// q_out fp32 [B][HQ][D]; out bf16 [B][ld_out] with q head h at columns
// h*D..h*D+D-1.  Partials (split > 1) fp32 [B][HQ][split][D + 4] = (acc, m, l).
//
// Attention runs one workgroup per (batch row, kv head, split), so the G =
// HQ/HKV query heads sharing a kv head read its keys and values once.  Its
// waves take 16-position blocks in turn:
//   scores   v_mfma_f32_16x16x32_bf16 over key rows and query rows; q is
//            carried as bf16 hi + lo parts (two MFMAs, ~16 significant bits;
//            an fp32 cache also splits k)
//   softmax  online (running max m, sum l) per head, exp2-based
//   p v      bf16 cache, D <= 256 (attn_bf16): v_mfma_f32_16x16x16_bf16 per
//            16 columns, p as bf16 hi + lo; fp32 cache or D = 512
//            (attn_kernel): VALU, lane l owns D/64 consecutive columns of
//            every head and reads each value row with one coalesced load
// The waves' (m, l, acc) are merged through LDS in a fixed order.
#include <algorithm>

#include "bz_attn.h"
#include "bz_device.h"

namespace bz {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// D = A B + C, 16x16x32: A[i][k] in lane i + 16 (k/8) element k%8, B[k][j]
// in lane j + 16 (k/8) element k%8, D[i][j] in lane j + 16 (i/4) element i%4.
__device__ __forceinline__ f32x4_t mfma16(const u32x4 a, const u32x4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                  c, 0, 0, 0);
}

typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// D = A B + C, 16x16x16: A[i][k] in lane i + 16 (k/4) element k%4, B[k][j]
// in lane j + 16 (k/4) element k%4, D[i][j] in lane j + 16 (i/4) element i%4
// (checked on the hardware).
__device__ __forceinline__ f32x4_t mfma16k16(const u32x2 a, const u32x2 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(bf16x4_t, a), __builtin_bit_cast(bf16x4_t, b),
                                                    c, 0, 0, 0);
}

__device__ __forceinline__ float ld_any(const void* p, bool f32, int64_t i) {
    return f32 ? reinterpret_cast<const float*>(p)[i] : bf16_to_f32(reinterpret_cast<const uint16_t*>(p)[i]);
}

// Raw bits of element i of a bf16 (BZ_DT_BF16), fp32 (BZ_DT_F32) or bool
// (BZ_MASK_BOOL) array, widened later by raw_f32: keeping the conversion
// away from the load lets the loads issued before and after it stay in
// flight.
__device__ __forceinline__ uint32_t ld_raw(const void* p, int kind, int64_t i) {
    if (kind == BZ_DT_F32) return reinterpret_cast<const uint32_t*>(p)[i];
    if (kind == BZ_MASK_BOOL) return reinterpret_cast<const uint8_t*>(p)[i];
    return reinterpret_cast<const uint16_t*>(p)[i];
}

// Element i of such an array without a branch on the type (ld_elem), and its
// value once the dword is there.
__device__ __forceinline__ RawWord ld_word(const void* p, int kind, int64_t i) {
    return ld_elem(p, kind == BZ_DT_F32 ? 2 : (kind == BZ_MASK_BOOL ? 0 : 1), i);
}
__device__ __forceinline__ float word_f32(RawWord r, int kind) {
    const uint32_t raw = r.w >> r.shift;
    const float num = __uint_as_float(kind == BZ_DT_F32 ? raw : raw << 16);
    const float allow = raw & 0xFFu ? 0.0f : -1e30f;
    return kind == BZ_MASK_BOOL ? allow : num;
}

// bf16 / fp32 as a value; a bool mask entry as additive (nonzero = attend
// -> 0, zero -> -1e30, the reference's conversion).
__device__ __forceinline__ float raw_f32(uint32_t v, int kind) {
    if (kind == BZ_DT_F32) return __uint_as_float(v);
    if (kind == BZ_MASK_BOOL) return v ? 0.0f : -1e30f;
    return __uint_as_float(v << 16);
}

__device__ __forceinline__ void st_any(void* p, bool f32, int64_t i, float v) {
    if (f32)
        reinterpret_cast<float*>(p)[i] = v;
    else
        reinterpret_cast<uint16_t*>(p)[i] = f32_to_bf16(v);
}

// Eight floats as bf16 hi + lo parts (x = hi + lo to ~16 significant bits).
__device__ __forceinline__ void split8(const float (&v)[8], u32x4& hi, u32x4& lo) {
    uint32_t h[4], l[4];
    for (int i = 0; i < 4; ++i) {
        const uint16_t h0 = f32_to_bf16(v[2 * i]), h1 = f32_to_bf16(v[2 * i + 1]);
        h[i] = (uint32_t)h0 | ((uint32_t)h1 << 16);
        l[i] = pack_bf16x2(v[2 * i] - bf16_to_f32(h0), v[2 * i + 1] - bf16_to_f32(h1));
    }
    hi = u32x4{h[0], h[1], h[2], h[3]};
    lo = u32x4{l[0], l[1], l[2], l[3]};
}

// Sum over the 64 lanes, every lane gets it: each 16-lane row by DPP, then
// rows 0..3 in order (the same order in every kernel of this file).
__device__ __forceinline__ float row_sum16(float v) {
    v += dpp_f32<kDppXor1>(v);
    v += dpp_f32<kDppXor2>(v);
    v += dpp_f32<0x124>(v);  // row_ror:4
    return v + dpp_f32<0x128>(v);  // row_ror:8
}

__device__ __forceinline__ float wave_sum64(float v) {
    v = row_sum16(v);
    const int bits = __float_as_int(v);
    return ((__int_as_float(__builtin_amdgcn_readlane(bits, 0)) + __int_as_float(__builtin_amdgcn_readlane(bits, 16))) +
            __int_as_float(__builtin_amdgcn_readlane(bits, 32))) +
           __int_as_float(__builtin_amdgcn_readlane(bits, 48));
}

// ---------------------------------------------------------------------------
// q/k RMSNorm + RoPE + cache write.  One workgroup per (batch row b, head h);
// heads [0, HQ) are queries, [HQ, HQ + HKV) key/value pairs.
// ---------------------------------------------------------------------------
constexpr int kRopeThreads = 256;
constexpr int kMaxRopeDim = 1024;

__global__ void __launch_bounds__(kRopeThreads) qkv_rope_cache_kernel(
    const uint16_t* qkv, int64_t ld_qkv, int HQ, int HKV, int D, const uint16_t* qn, const uint16_t* kn, float eps,
    const void* cosp, const void* sinp, bool cs_f32, int64_t ld_cs, const int64_t* pos_p, float* q_out, void* kc,
    void* vc, int S, bool cache_f32, int64_t* seq_len) {
    __shared__ float vals[kMaxRopeDim];
    __shared__ float part[kRopeThreads / 64];
    const int b = blockIdx.x, h = blockIdx.y;
    const bool is_q = h < HQ;
    const uint16_t* src = qkv + (int64_t)b * ld_qkv + (int64_t)h * D;
    const uint16_t* nw = is_q ? qn : kn;
    float ss = 0.0f;
    for (int d = threadIdx.x; d < D; d += kRopeThreads) {
        const float v = bf16_to_f32(src[d]);
        vals[d] = v;
        ss += v * v;
    }
    ss = wave_sum64(ss);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
    __syncthreads();
    float inv = 1.0f;
    if (nw) {
        float t = 0.0f;
        for (int w = 0; w < kRopeThreads / 64; ++w) t += part[w];
        inv = 1.0f / sqrtf(t / (float)D + eps);
    }
    const int half = D >> 1;
    const int64_t cs = (int64_t)b * ld_cs;
    const int64_t pos = *pos_p;
    if (seq_len && b == 0 && h == 0 && threadIdx.x == 0) *seq_len = pos + 1;
    // a position outside the cache writes no cache entry
    if (!is_q && (pos < 0 || pos >= S)) return;
    for (int d = threadIdx.x; d < D; d += kRopeThreads) {
        // rotate_half(v) = [-v2, v1]
        const int dp = d < half ? d + half : d - half;
        float v = vals[d], r = vals[dp];
        if (nw) {
            v = v * inv * bf16_to_f32(nw[d]);
            r = r * inv * bf16_to_f32(nw[dp]);
        }
        if (d < half) r = -r;
        const float o = v * ld_any(cosp, cs_f32, cs + d) + r * ld_any(sinp, cs_f32, cs + d);
        if (is_q) {
            q_out[((int64_t)b * HQ + h) * D + d] = o;
        } else {
            const int64_t base = (((int64_t)b * HKV + (h - HQ)) * S + pos) * D;
            st_any(kc, cache_f32, base + d, o);
            st_any(vc, cache_f32, base + d, bf16_to_f32(src[(int64_t)HKV * D + d]));
        }
    }
}

// ---------------------------------------------------------------------------
// Decode attention: one workgroup per (batch row b, kv head j, split sp).
// ---------------------------------------------------------------------------
constexpr int kBlk = 16;           // positions per block (the MFMA's 16 columns)
constexpr int kUnsplitMax = 160;   // attended positions up to which attn_kernel runs unsplit
constexpr float kNegBig = -1e30f;  // initial running max, as the reference
constexpr float kLog2e = 1.4426950408889634f;

// 2^x with the hardware instruction alone (results below 2^-126 flush to
// zero, which a softmax weight can afford).
__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }

struct AttnParams {
    // fused step: the token's qkv row and the q/k norm + RoPE inputs
    const uint16_t* qkv;
    int64_t ld_qkv;
    const uint16_t* qn;
    const uint16_t* kn;
    float eps;
    const void* cosp;
    const void* sinp;
    int cs_f32;
    int64_t ld_cs;
    int64_t* seq_len;
    // attention only: q already normed and rotated, fp32 [B][HQ][D]
    const float* q;
    void* kc;
    void* vc;
    const void* mask;
    int64_t ld_mask;
    int mask_dtype;
    const int64_t* pos;
    float scale;
    int HQ, HKV, G, S, split;
    int split_cap;       // splits attn_bf16 uses at most: split, or one workgroup per CU
    float* part;         // [B][HQ][split][D + 4] (acc, m, l, 2 pad)
    unsigned* counters;  // [B][HKV] arrivals, zero between calls
    uint16_t* out;
    int64_t ld_out;
};

// attn_kernel's registers of one 16-position block: key operands and raw
// value words (lane l holds columns DL l .. DL l + DL - 1 of all 16 rows).
template <int DL, bool F32C>
struct KvBlock {
    static constexpr int T = 2 * DL;                                    // MFMA k-steps per key row
    static_assert(F32C || DL == 8, "bf16 caches of D <= 256 run on attn_bf16");
    static constexpr int VW = F32C ? DL : DL / 2;  // value words per row
    u32x4 kh[T], kl[T];
    uint32_t v[kBlk][VW];
    uint32_t mraw;  // raw mask entry at this lane's key position
};

// 8 cache elements of one key row as an MFMA operand; an fp32 cache gives
// hi + lo bf16 parts.
template <bool F32C>
__device__ __forceinline__ void load_k8(const void* kc, int64_t off, u32x4& hi, u32x4& lo) {
    if constexpr (F32C) {
        const float* p = reinterpret_cast<const float*>(kc) + off;
        const float4 x0 = *reinterpret_cast<const float4*>(p);
        const float4 x1 = *reinterpret_cast<const float4*>(p + 4);
        const float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
        split8(v, hi, lo);
    } else {
        hi = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(kc) + off);
        lo = u32x4{0u, 0u, 0u, 0u};
    }
}

// DL consecutive value elements of one row, as raw words.
template <int DL, bool F32C>
__device__ __forceinline__ void load_vraw(const void* vc, int64_t off, uint32_t (&w)[KvBlock<DL, F32C>::VW]) {
    if constexpr (F32C) {
        const uint32_t* p = reinterpret_cast<const uint32_t*>(vc) + off;
        if constexpr (DL >= 4) {
            for (int i = 0; i < DL; i += 4) {
                const u32x4 t = *reinterpret_cast<const u32x4*>(p + i);
                w[i] = t[0];
                w[i + 1] = t[1];
                w[i + 2] = t[2];
                w[i + 3] = t[3];
            }
        } else {
            for (int i = 0; i < DL; ++i) w[i] = p[i];
        }
    } else {
        const u32x4 t = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(vc) + off);
        for (int i = 0; i < 4; ++i) w[i] = t[i];
    }
}

template <int DL, bool F32C>
__device__ __forceinline__ float vword(const uint32_t (&w)[KvBlock<DL, F32C>::VW], int e) {
    if constexpr (F32C) return __uint_as_float(w[e]);
    return (e & 1) ? bf16_hi(w[e >> 1]) : bf16_lo(w[e >> 1]);
}

// One block's loads: key rows s0 + col (lane col), value rows s0 .. s0 + 15
// and the mask entries, rows past the split's last one clamped to it.  s0
// and s_hi are wave-uniform, so the value rows' addresses are scalar and
// each load carries only the lane's column offset.
template <int DL, bool F32C>
__device__ __forceinline__ void load_block(const AttnParams& a, int64_t kv_base, int s0, int s_hi, int64_t mrow,
                                           int lane, KvBlock<DL, F32C>& blk) {
    constexpr int D = 64 * DL;
    constexpr int ES = F32C ? 4 : 2;  // element bytes
    const int last = max(s_hi - 1, 0);  // an empty range reads row 0 (every cache has one), unused
    const int col = lane & 15, grp = lane >> 4;
    const int kpos = min(s0 + col, last);
    blk.mraw = ld_raw(a.mask, a.mask_dtype, mrow + kpos);  // first: its load depends on the dtype
    const char* kc = static_cast<const char*>(a.kc) + kv_base * ES;
    const char* krow = kc + (int64_t)kpos * (D * ES) + 8 * grp * ES;
    for (int t = 0; t < KvBlock<DL, F32C>::T; ++t) load_k8<F32C>(krow, 32 * t, blk.kh[t], blk.kl[t]);
    const char* vc = static_cast<const char*>(a.vc) + kv_base * ES;
    for (int p = 0; p < kBlk; ++p) {
        const int row = min(s0 + p, last);
        load_vraw<DL, F32C>(vc + (int64_t)row * (D * ES), DL * lane, blk.v[p]);
    }
}

// Max / sum over each aligned group of 16 lanes (one DPP row; every lane
// gets it): swap within pairs, within quads, then rotate the row by 4 and 8.
constexpr int kDppRowRor4 = 0x124, kDppRowRor8 = 0x128;

__device__ __forceinline__ float max16(float v) {
    v = fmaxf(v, dpp_f32<kDppXor1>(v));
    v = fmaxf(v, dpp_f32<kDppXor2>(v));
    v = fmaxf(v, dpp_f32<kDppRowRor4>(v));
    return fmaxf(v, dpp_f32<kDppRowRor8>(v));
}

__device__ __forceinline__ float sum16(float v) {
    v += dpp_f32<kDppXor1>(v);
    v += dpp_f32<kDppXor2>(v);
    v += dpp_f32<kDppRowRor4>(v);
    return v + dpp_f32<kDppRowRor8>(v);
}

__device__ __forceinline__ float bcast(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// The waves' state in LDS ([wave][GM heads], accumulator rows of ROW floats),
// behind a barrier, into the output or, over nsp > 1 splits, the workspace,
// whose last arrival combines them.  The first nact waves have state.
template <int D, int GM, int NWV, int ROW>
__device__ __forceinline__ void merge_and_combine(const AttnParams& a, int b, int j, int sp, int nsp, int nact, int tid,
                                                  const float* st_m, const float* st_l, const float* st_acc, int* last) {
    // Merge the waves in a fixed order; write the output or the partial.
    // Each thread forms its head's wave weights itself (8 values from LDS):
    // no serial step and no barrier between the state and the merge.
    constexpr int kThreads = 64 * NWV;
    const int G = a.G;
    const int64_t hq0 = (int64_t)b * a.HQ + (int64_t)j * G;
    for (int i = tid; i < G * D; i += kThreads) {
        const int h = i / D, d = i - h * D;
        float mt = kNegBig;
        for (int w = 0; w < nact; ++w) mt = fmaxf(mt, st_m[w * GM + h]);
        float lt = 0.0f, at = 0.0f;
        for (int w = 0; w < nact; ++w) {
            const float f = fexp2((st_m[w * GM + h] - mt) * kLog2e);
            lt += st_l[w * GM + h] * f;
            at += st_acc[(w * GM + h) * ROW + d] * f;
        }
        if (nsp == 1) {
            a.out[(int64_t)b * a.ld_out + (int64_t)(j * G + h) * D + d] = f32_to_bf16(lt > 0.0f ? at / lt : 0.0f);
        } else {  // agent-scope stores: coherent across XCDs without an L2 write-back
            float* pp = a.part + ((hq0 + h) * a.split + sp) * (D + 4);
            __hip_atomic_store(&pp[d], at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (d == 0) {
                __hip_atomic_store(&pp[D], mt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(&pp[D + 1], lt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
    if (nsp == 1) return;

    // The last workgroup of (b, j) to finish combines the splits.  Every
    // thread waits until its partial stores have completed (agent-scope
    // stores complete at the point of coherence) before the workgroup counts
    // its arrival; the last one reads the partials with agent-scope loads.
    // No L2 write-back or invalidate is needed for that.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
        const unsigned prev =
            __hip_atomic_fetch_add(&a.counters[b * a.HKV + j], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *last = prev == (unsigned)nsp - 1u;
    }
    __syncthreads();
    if (!*last) return;
    // Element i = (h, d): each thread loads, for its NE elements, every
    // split's partial and its head's (m, l) in batches of SB splits (all in
    // flight at once; SB NE <= 16 keeps them in registers), and merges them
    // in split order, online: with M the running max, acc and L are rescaled
    // by exp(M_old - M) and gain w_s acc_s and w_s l_s, w_s = exp(m_s - M).
    // One memory round trip per batch and no barrier (the weights were first
    // formed per head in LDS: a second round trip and a barrier).
    constexpr int NE = (GM * D + kThreads - 1) / kThreads;
    constexpr int SB = NE <= 2 ? 8 : (NE <= 4 ? 4 : (NE <= 8 ? 2 : 1));
    float acc0[NE], lsum[NE], mrun[NE];
    for (int q = 0; q < NE; ++q) {
        acc0[q] = 0.0f;
        lsum[q] = 0.0f;
        mrun[q] = kNegBig;
    }
    for (int s0 = 0; s0 < nsp; s0 += SB) {
        float v[NE][SB], ms[NE][SB], ls[NE][SB];
        for (int q = 0; q < NE; ++q) {
            const int i = min(tid + q * kThreads, G * D - 1);
            const int h = i / D, d = i - h * D;
            const float* ph = a.part + (hq0 + h) * a.split * (D + 4);
            for (int u = 0; u < SB; ++u) {
                const float* pp = ph + min(s0 + u, nsp - 1) * (D + 4);
                v[q][u] = __hip_atomic_load(pp + d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                ms[q][u] = __hip_atomic_load(pp + D, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                ls[q][u] = __hip_atomic_load(pp + D + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        for (int q = 0; q < NE; ++q) {
            float mb = mrun[q];
            for (int u = 0; u < SB; ++u)
                if (s0 + u < nsp) mb = fmaxf(mb, ms[q][u]);
            const float rs = fexp2((mrun[q] - mb) * kLog2e);
            acc0[q] *= rs;
            lsum[q] *= rs;
            mrun[q] = mb;
            for (int u = 0; u < SB; ++u)
                if (s0 + u < nsp) {
                    const float w = fexp2((ms[q][u] - mb) * kLog2e);
                    acc0[q] += v[q][u] * w;
                    lsum[q] += ls[q][u] * w;
                }
        }
    }
    for (int q = 0; q < NE; ++q) {
        const int i = tid + q * kThreads;
        if (i < G * D) {
            const int h = i / D, d = i - h * D;
            const float lt = lsum[q];
            a.out[(int64_t)b * a.ld_out + (int64_t)(j * G + h) * D + d] =
                f32_to_bf16(lt > 0.0f ? acc0[q] / lt : 0.0f);
        }
    }
    if (tid == 0) __hip_atomic_store(&a.counters[b * a.HKV + j], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------------------
// Decode attention over a bf16 cache, D = 64, 128 or 256: one workgroup per
// (batch row b, kv head j, split sp), its waves taking 16-position blocks.
//
// Bound by latency: a step attends a few hundred positions, so each wave has
// one or two blocks and the chain launch, loads, q, scores, softmax, p v,
// merge is what it takes.  Hence
//   * one barrier before the blocks: a wave norms and rotates a whole q or k
//     head by itself (its sum of squares by DPP, the rotary partner column in
//     the same lane) and writes it to LDS as the MFMA operand's hi and lo
//     bf16 parts; the new key and value reach the block that holds them
//     through LDS too, not through the cache;
//   * the scores transposed, A = 16 key rows, B = the G <= 16 query heads:
//     lane (head, grp) gets positions 4 grp .. 4 grp + 3, which is exactly the B
//     operand of p v on v_mfma_f32_16x16x16_bf16 (A = the transposed value
//     rows), so p never leaves its lane; a head's max and sum over the
//     positions are two lane-row swaps (v_permlane32_swap, v_permlane16_swap);
//   * the first workgroup of a (row, kv head) issues its first blocks' loads
//     before it knows the position: block wave + NW sp is its first whatever
//     the number of splits in use.
//   * loads whose element type is a run-time argument (mask, cos, sin) take the
//     aligned dword: a branch on the type put a wait for everything in flight
//     at its end.
// Measured on MI355X (cold caches, graph replays, default split) against the
// kernel with four prologue barriers, scores not transposed and p through
// LDS: 8 / 2 heads of 128, B = 2, 17 positions 5.25 -> 4.25 us; 16 / 8 heads of
// 128, B = 2, 612 of 1024 positions 8.55 -> 7.68; 16 / 4 heads of 256, B = 2,
// 128 positions 8.71 -> 7.77, 1902 of 2048 13.96 -> 12.94.  Every sum keeps that
// kernel's order (norm: 64 columns over the lanes, then in column order; scores:
// hi and lo in one chain; l: 16 positions as sum16 adds them), so an unsplit
// step gives the same bits: tokens are picked from what it feeds.
// ---------------------------------------------------------------------------
template <int DL>
struct KvRows {
    u32x4 k[2 * DL];         // key row `col`, elements 32 t + 8 grp + 0..7
    uint32_t v[4][2 * DL];   // value rows 4 grp + r, columns v_col(c, col) of attn_bf16, c = 0..4 DL - 1
    RawWord mraw[4];         // mask entries of positions 4 grp + r
};

// Reduce over the four 16-lane rows of a wave; every lane gets the result of
// its column.
template <typename F>
__device__ __forceinline__ float across_rows(float v, F f) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    const float t = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(t), __float_as_uint(t), false, false);
    return f(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// The four rows' values of a column, in every lane of it.
__device__ __forceinline__ void all_rows(float v, float (&o)[4]) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    const auto lo = __builtin_amdgcn_permlane16_swap(a[0], a[0], false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(a[1], a[1], false, false);
    o[0] = __uint_as_float(lo[0]);
    o[1] = __uint_as_float(lo[1]);
    o[2] = __uint_as_float(hi[0]);
    o[3] = __uint_as_float(hi[1]);
}

// attended positions up to which attn_bf16 runs unsplit (figures at nsp below)
__host__ __device__ constexpr int attn_unsplit(int DL) { return DL == 4 ? 224 : 256; }

template <int DL, int GM, bool FUSED, int NWV>
__global__ void __launch_bounds__(64 * NWV) attn_bf16(const void* hrows, const void* hcos, const void* hsin,
                                                      const int64_t* hpos, void* hkc, void* hvc, int hld_qkv,
                                                      uint32_t hshape, AttnParams a) {
    constexpr int D = 64 * DL, T = 2 * DL, NT = 4 * DL;
    // column of operand row i of p v's tile c: lanes read value rows in runs
    // of 16 bytes side by side (with each lane's columns contiguous, a 256-wide
    // row took two half-used passes over its lines)
    auto v_col = [](int c, int i) { return DL == 1 ? 4 * i + c : 128 * (c >> 3) + 8 * i + (c & 7); };
    constexpr int kAccRow = D + 4;  // floats of one head's partial (16-byte rows, off the bank period)
    __shared__ u32x4 qop[T][2][64];             // B operands of the query heads: hi, lo
    __shared__ __attribute__((aligned(16))) uint16_t knew[D], vnew[D];  // the new token's key and value
    __shared__ float st_m[NWV][GM], st_l[NWV][GM];
    __shared__ __attribute__((aligned(16))) float st_acc[NWV][GM][kAccRow];
    __shared__ int last;
    const int b = blockIdx.x, j = blockIdx.y, sp = blockIdx.z;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, grp = lane >> 4;
    const int G = hshape & 31u, HKV = (hshape >> 5) & 0xFFFFu, HQ = G * HKV;

    const int64_t pos = *hpos;

    // 1. raw rows of the prologue: row r = wave + NWV i is query head j G + r
    //    (r < G), the key head (r = G) or the value head (G + 1); lane l holds
    //    columns l + 64 e.  Rows past the last read as zeros without requests.
    constexpr int NR = FUSED ? GM + 2 : GM, NI = (NR + NWV - 1) / NWV;
    const int nrows = FUSED ? G + 2 : G;
    uint32_t raw[NI][DL], nw[NI][DL];
    RawWord cs[DL], sn[DL];
    const int cs_kind = hshape >> 21 & 1u ? BZ_DT_F32 : BZ_DT_BF16;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int r = wave + NWV * i;
        if constexpr (FUSED) {
            const int head = r < G ? j * G + r : (r == G ? HQ + j : HQ + HKV + j);
            const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(
                static_cast<const uint16_t*>(hrows) + (int64_t)b * hld_qkv + (int64_t)(r < nrows ? head : 0) * D,
                r < nrows ? (uint32_t)D * 2u : 0u);
#pragma unroll
            for (int e = 0; e < DL; ++e) raw[i][e] = __builtin_amdgcn_raw_buffer_load_b16(rs, (lane + 64 * e) * 2, 0, 0);
        } else {
            const __amdgpu_buffer_rsrc_t rs =
                buffer_rsrc(static_cast<const float*>(hrows) + ((int64_t)b * HQ + (int64_t)j * G + (r < nrows ? r : 0)) * D,
                            r < nrows ? (uint32_t)D * 4u : 0u);
#pragma unroll
            for (int e = 0; e < DL; ++e) raw[i][e] = buffer_ld4(rs, (lane + 64 * e) * 4);
        }
    }
    if constexpr (FUSED) {
        const int64_t c0 = hshape >> 22 & 1u ? 0 : (int64_t)b * a.ld_cs;
#pragma unroll
        for (int e = 0; e < DL; ++e) {
            cs[e] = ld_word(hcos, cs_kind, c0 + lane + 64 * e);
            sn[e] = ld_word(hsin, cs_kind, c0 + lane + 64 * e);
        }
        // (everything so far needs preloaded arguments only)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int r = wave + NWV * i;
            const uint16_t* w = r < G ? a.qn : a.kn;  // without norm weights or past the normed rows: an empty range
            const __amdgpu_buffer_rsrc_t ws = buffer_rsrc(w, w && r <= G ? (uint32_t)D * 2u : 0u);
#pragma unroll
            for (int e = 0; e < DL; ++e) nw[i][e] = __builtin_amdgcn_raw_buffer_load_b16(ws, (lane + 64 * e) * 2, 0, 0);
        }
    }

    // 2. the wave's first block.  Rows past the cache read as zeros; rows past
    //    the attended range are loaded as they are and dropped below.
    const int64_t kv_base = ((int64_t)b * HKV + j) * a.S * D;
    const uint32_t kv_bytes = (uint32_t)a.S * (D * 2);  // S D 4 < 2^32 (checked at set-up)
    const int64_t mrow = (int64_t)b * a.ld_mask;
    auto load_rows = [&](KvRows<DL>& blk, int s0, uint32_t bytes) {
        const __amdgpu_buffer_rsrc_t kr = buffer_rsrc(static_cast<const uint16_t*>(hkc) + kv_base, bytes);
        const __amdgpu_buffer_rsrc_t vr = buffer_rsrc(static_cast<const uint16_t*>(hvc) + kv_base, bytes);
#pragma unroll
        for (int r = 0; r < 4; ++r) blk.mraw[r] = ld_word(a.mask, a.mask_dtype, mrow + min(s0 + 4 * grp + r, a.S - 1));
        const uint32_t ko = (uint32_t)(s0 + col) * (D * 2) + 16 * grp;
#pragma unroll
        for (int t = 0; t < T; ++t) blk.k[t] = buffer_ld16(kr, ko + 64 * t);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t vo = (uint32_t)(s0 + 4 * grp + r) * (D * 2) + (DL == 1 ? 8 : 16) * col;
            if constexpr (DL == 1) {
                const u32x2 t = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(vr, vo, 0, 0));
                blk.v[r][0] = t[0];
                blk.v[r][1] = t[1];
            } else {
#pragma unroll
                for (int i = 0; i < DL / 2; ++i) {
                    const u32x4 t = buffer_ld16(vr, vo + 256 * i);
#pragma unroll
                    for (int e = 0; e < 4; ++e) blk.v[r][4 * i + e] = t[e];
                }
            }
        }
    };
    // cache positions [0, min(pos, S - 1)]; none for pos < 0 (output 0)
    const int kv_len = pos < 0 ? 0 : (pos >= a.S ? a.S : (int)pos + 1);
    const int nblk = (kv_len + kBlk - 1) / kBlk;
    // Splits in use (decided from the device position, so a captured graph
    // follows it): none while two blocks per wave cover the positions, else
    // as many as have a block for every wave, and no more workgroups than
    // CUs (more are not launched); of those launched, the ones that the
    // position leaves without a range leave before any barrier.  Measured on MI355X, unsplit
    // against 8 splits: D = 128 (16 / 8 heads, B = 2) 7.54 / 7.09 us at 331
    // positions (6.56 / 7.02 at 256 when both could be forced); D = 256 (16 / 4
    // heads, B = 1) 8.69 / 8.78 at 160, 10.63 / 10.22 at 256.  64 (row, kv head)
    // pairs at 2001 positions: 4 splits 16.5 us, 5 21.8, 8 19.5, 16 25.8.  Above
    // 128 pairs one split is left; against the kernel named
    // above at 16 splits (16 / 8 heads of 128, 1902 of 2048 positions): 96 pairs
    // 28.2 -> 22.0 us, 136 37.7 -> 29.7, 200 43.1 -> 30.5, 256 54.6 -> 38.4.
    const int nsp = kv_len <= attn_unsplit(DL) ? 1 : min(a.split_cap, (nblk + NWV - 1) / NWV);
    KvRows<DL> cur;
    int s0 = (sp * NWV + wave) * kBlk;
    uint32_t live = kv_bytes;
    if (sp != 0) {  // split 0 does not wait for the position here
        if (sp >= nsp) return;
        if (s0 >= kv_len) live = 0u;
    }
    load_rows(cur, s0, live);

    const int new_blk = FUSED && pos >= 0 && pos < a.S ? (int)pos / kBlk : -1;  // holds the new token
    const bool has_new = new_blk >= 0 && (new_blk / NWV) % nsp == sp;

    // 3. each wave's rows: norm, rotate, to LDS
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int r = wave + NWV * i;
        if (r >= nrows) continue;
        float v[DL];
        if constexpr (FUSED) {
            if (r == G + 1) {
                if (has_new) {
#pragma unroll
                    for (int e = 0; e < DL; ++e) {
                        const int d = lane + 64 * e;
                        vnew[d] = (uint16_t)raw[i][e];
                        static_cast<uint16_t*>(hvc)[kv_base + pos * D + d] = (uint16_t)raw[i][e];
                    }
                }
                continue;
            }
            float ss = 0.0f;  // each 64 columns over the lanes, then in column order
#pragma unroll
            for (int e = 0; e < DL; ++e) {
                v[e] = __uint_as_float(raw[i][e] << 16);
                ss += wave_sum64(v[e] * v[e]);
            }
            if (a.qn) {
                const float inv = 1.0f / sqrtf(ss / (float)D + a.eps);
#pragma unroll
                for (int e = 0; e < DL; ++e) v[e] = v[e] * inv * __uint_as_float(nw[i][e] << 16);
            }
            // rotate_half(v) = [-v2, v1]; the partner column d +- D/2 is in
            // this lane (D >= 128) or 32 lanes away (D = 64)
            float o[DL];
#pragma unroll
            for (int e = 0; e < DL; ++e) {
                float rr;
                if constexpr (DL == 1) {
                    rr = __shfl_xor(v[0], 32, 64);
                    if (lane < 32) rr = -rr;
                } else {
                    rr = e < DL / 2 ? -v[e + DL / 2] : v[e - DL / 2];
                }
                o[e] = v[e] * word_f32(cs[e], cs_kind) + rr * word_f32(sn[e], cs_kind);
            }
            if (r == G) {
                if (has_new) {
#pragma unroll
                    for (int e = 0; e < DL; ++e) {
                        const int d = lane + 64 * e;
                        const uint16_t h = f32_to_bf16(o[e]);
                        knew[d] = h;
                        static_cast<uint16_t*>(hkc)[kv_base + pos * D + d] = h;
                    }
                }
                continue;
            }
#pragma unroll
            for (int e = 0; e < DL; ++e) v[e] = o[e];
        } else {
#pragma unroll
            for (int e = 0; e < DL; ++e) v[e] = __uint_as_float(raw[i][e]);
        }
        // element d of head r: step d / 32, lane r + 16 ((d / 8) % 4), element d % 8
        uint16_t* q16 = reinterpret_cast<uint16_t*>(&qop[0][0][0]);
#pragma unroll
        for (int e = 0; e < DL; ++e) {
            const int d = lane + 64 * e;
            const int at = ((d >> 5) * 2 * 64 + r + 16 * ((d >> 3) & 3)) * 8 + (d & 7);
            const float x = v[e] * a.scale;
            const uint16_t h = f32_to_bf16(x);
            q16[at] = h;
            q16[at + 64 * 8] = f32_to_bf16(x - bf16_to_f32(h));
        }
    }
    if (FUSED && a.seq_len && b == 0 && j == 0 && sp == 0 && tid == 0) *a.seq_len = pos + 1;
    __syncthreads();

    // 4. the wave's blocks: lane (col, grp) holds head col's scores at
    //    positions 4 grp + r; m is the head's running max (the same in its
    //    four lanes), l[r] the sum of its position's weights, acc[c][r] the head's
    //    output at column v_col(c, 4 grp + r)
    float m = kNegBig, l[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4_t acc[NT];
#pragma unroll
    for (int c = 0; c < NT; ++c) acc[c] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    const bool any = s0 < kv_len;
    auto process = [&](KvRows<DL>& cur, int s0) __attribute__((always_inline)) {
        if (has_new && s0 == new_blk * kBlk) {  // uniform: the new token's rows from LDS
            const int at = (int)pos - s0;
            u32x4 kn[T];
            uint32_t vn[2 * DL];
#pragma unroll
            for (int t = 0; t < T; ++t) kn[t] = *reinterpret_cast<const u32x4*>(&knew[32 * t + 8 * grp]);
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q) cur.k[t][q] = col == at ? kn[t][q] : cur.k[t][q];
            if constexpr (DL == 4) __builtin_amdgcn_sched_barrier(0);  // the registers of both do not fit at once
#pragma unroll
            for (int i = 0; i < 2 * DL; ++i) vn[i] = *reinterpret_cast<const uint32_t*>(&vnew[v_col(2 * i, col)]);
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int i = 0; i < 2 * DL; ++i) cur.v[r][i] = 4 * grp + r == at ? vn[i] : cur.v[r][i];
        }
        f32x4_t sc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < T; ++t) {
            sc = mfma16(cur.k[t], qop[t][0][lane], sc);
            sc = mfma16(cur.k[t], qop[t][1][lane], sc);
        }
        float s[4], bm = kNegBig;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const bool valid = s0 + 4 * grp + r < kv_len;
            s[r] = valid ? sc[r] + word_f32(cur.mraw[r], a.mask_dtype) : kNegBig;
            bm = fmaxf(bm, s[r]);
            // (a value row past the range may hold anything)
#pragma unroll
            for (int i = 0; i < 2 * DL; ++i) cur.v[r][i] = valid ? cur.v[r][i] : 0u;
        }
        const float mn = fmaxf(m, across_rows(bm, [](float x, float y) { return fmaxf(x, y); }));
        const float alpha = fexp2((m - mn) * kLog2e);
        m = mn;
        float p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            p[r] = s0 + 4 * grp + r < kv_len ? fexp2((s[r] - mn) * kLog2e) : 0.0f;
            l[r] = l[r] * alpha + p[r];
        }
        const uint32_t h01 = pack_bf16x2(p[0], p[1]), h23 = pack_bf16x2(p[2], p[3]);
        const u32x2 ph = {h01, h23};
        const u32x2 pl = {pack_bf16x2(p[0] - bf16_lo(h01), p[1] - bf16_hi(h01)),
                          pack_bf16x2(p[2] - bf16_lo(h23), p[3] - bf16_hi(h23))};
#pragma unroll
        for (int c = 0; c < NT; ++c) {
            // A: column v_col(c, col) of value rows 4 grp .. 4 grp + 3
            const uint32_t w0 = cur.v[0][c >> 1], w1 = cur.v[1][c >> 1], w2 = cur.v[2][c >> 1], w3 = cur.v[3][c >> 1];
            const uint32_t sel = c & 1 ? 0x07060302u : 0x05040100u;  // high or low halves of a pair of rows
            const u32x2 av = {__builtin_amdgcn_perm(w1, w0, sel), __builtin_amdgcn_perm(w3, w2, sel)};
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[c][r] *= alpha;
            acc[c] = mfma16k16(av, ph, acc[c]);
            acc[c] = mfma16k16(av, pl, acc[c]);
        }
    };
    // (the first block by itself: behind a loop the waits for its key rows
    // would also wait for its value rows)
    if (any) process(cur, s0);
    for (s0 += nsp * NWV * kBlk; s0 < kv_len; s0 += nsp * NWV * kBlk) {
        load_rows(cur, s0, kv_bytes);
        process(cur, s0);
    }

    // 5. the waves' state to LDS, merged in wave order; a wave past the
    //    positions has none
    const int nact = min(NWV, nblk - sp * NWV);  // <= 0 only without any position
    if (any) {
        float ql[4];
        all_rows((l[0] + l[1]) + (l[2] + l[3]), ql);
        if (col < G) {
            if (grp == 0) {
                st_m[wave][col] = m;
                st_l[wave][col] = (ql[0] + ql[3]) + (ql[2] + ql[1]);  // the order of sum16
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int c = 0; c < NT; c += 4)
                    *reinterpret_cast<float4*>(&st_acc[wave][col][v_col(c, 4 * grp + r)]) =
                        make_float4(acc[c][r], acc[c + 1][r], acc[c + 2][r], acc[c + 3][r]);
        }
    }
    __syncthreads();
    merge_and_combine<D, GM, NWV, kAccRow>(a, b, j, sp, nsp, nact, tid, &st_m[0][0], &st_l[0][0], &st_acc[0][0][0], &last);
}

// DL = D / 64 columns per lane; GM = 4 or 16 heads of register state (G <=
// GM); F32C: fp32 cache; FUSED: q (and the new k, v) computed from qkv.
constexpr int kAttnWaves = 4;
template <int DL, int GM, bool F32C, bool FUSED>
__global__ void __launch_bounds__(64 * kAttnWaves) attn_kernel(const void* hrows, const void* hcos, const void* hsin,
                                                        const int64_t* hpos, void* hkc, void* hvc, int hld_qkv, int hG,
                                                        AttnParams a) {
    // the fields of the first loads, preloaded into SGPRs at wave launch
    // (kernarg preloading, as for the GEMV kernels); the host passes the same
    // values in the struct
    if constexpr (FUSED)
        a.qkv = static_cast<const uint16_t*>(hrows);
    else
        a.q = static_cast<const float*>(hrows);
    a.cosp = hcos;
    a.sinp = hsin;
    a.pos = hpos;
    a.kc = hkc;
    a.vc = hvc;
    a.ld_qkv = hld_qkv;
    a.G = hG;
    constexpr int kAttnThreads = 64 * kAttnWaves;
    constexpr int D = 64 * DL;
    constexpr int T = D / 32;
    using Blk = KvBlock<DL, F32C>;
    __shared__ float qf[GM][D];
    __shared__ float css[(GM + 2) * DL];
    __shared__ float rinv[GM + 1];
    __shared__ u32x4 qop[T][2][64];  // the A operand (q hi, lo) of every lane
    __shared__ float p_lds[kAttnWaves][kBlk * GM];  // [position][head]
    __shared__ float st_m[kAttnWaves][GM], st_l[kAttnWaves][GM];
    __shared__ float st_acc[kAttnWaves][GM][D];  // also the raw qkv rows of the prologue
    __shared__ int last;

    const int b = blockIdx.x, j = blockIdx.y, sp = blockIdx.z;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: block starts are scalar
    const int G = a.G;
    const int col = lane & 15, grp = lane >> 4;

    // The query rows (FUSED: the token's q heads j*G.., its key head j and
    // value head j) go out first, as raw words, one element per thread and
    // row chunk; nothing here waits on the cache position.
    constexpr int NR = FUSED ? GM + 2 : GM;                            // rows at most
    constexpr int NI = (NR * D + kAttnThreads - 1) / kAttnThreads;     // elements per thread
    const int nrows = FUSED ? G + 2 : G;
    uint32_t pre[NI];
    // (every thread issues all NI loads, rows past the last clamped to it,
    // so the number of loads in flight never depends on a branch)
    for (int i = 0; i < NI; ++i) {
        const int e = tid + i * kAttnThreads;
        const int r = min(e / D, nrows - 1), d = e % D;
        if constexpr (FUSED) {
            const int head = r < G ? j * G + r : (r == G ? a.HQ + j : a.HQ + a.HKV + j);
            pre[i] = a.qkv[(int64_t)b * a.ld_qkv + (int64_t)head * D + d];
        } else {
            pre[i] = __float_as_uint(a.q[((int64_t)b * a.HQ + (int64_t)j * G + r) * D + d]);
        }
    }

    // RoPE and norm operands of this thread's columns: element e = tid +
    // 256 i of a row sits in column (tid + 256 i) % D, i.e. column tid % D
    // for D <= 256 and tid or tid + 256 (i even / odd) for D = 512.
    constexpr int NC = D > kAttnThreads ? 2 : 1;
    const int cs_kind = a.cs_f32 ? BZ_DT_F32 : BZ_DT_BF16;
    uint32_t cs_r[NC], sn_r[NC], nw_r[NC][4];  // cos, sin, q/k norm weights at d and its partner
    if constexpr (FUSED) {
        const int64_t cs = (int64_t)b * a.ld_cs;
        for (int c = 0; c < NC; ++c) {
            const int d = (tid + c * kAttnThreads) % D;
            const int dp = d < D / 2 ? d + D / 2 : d - D / 2;
            cs_r[c] = ld_raw(a.cosp, cs_kind, cs + d);
            sn_r[c] = ld_raw(a.sinp, cs_kind, cs + d);
            // without norm weights, in-bounds loads of cos stand in (unused)
            const uint16_t* qn = a.qn ? a.qn : static_cast<const uint16_t*>(a.cosp);
            const uint16_t* kn = a.qn ? a.kn : static_cast<const uint16_t*>(a.cosp);
            nw_r[c][0] = qn[d];
            nw_r[c][1] = qn[dp];
            nw_r[c][2] = kn[d];
            nw_r[c][3] = kn[dp];
        }
    }

    // cache positions [0, min(pos, S - 1)]; none for pos < 0 (output 0)
    const int64_t pos = *a.pos;
    const int kv_len = pos < 0 ? 0 : (pos >= a.S ? a.S : (int)pos + 1);
    // Short contexts run unsplit: the workgroup of split 0 takes every
    // position and writes the output itself; the others leave before any
    // barrier.  Up to about 160 positions that beats a split plus the
    // cross-workgroup combine (measured on MI355X over bf16 caches, 16 q / 4 kv
    // heads of 256: unsplit 8.5 against 9.7 us at 128 positions, even at 160,
    // split 9.9 against 10.2 us at 192).  The choice follows the device position, so a
    // captured graph adapts to it.
    const int nsp = kv_len <= kUnsplitMax ? 1 : a.split;
    if (sp >= nsp) return;
    const int per = (kv_len + nsp - 1) / nsp;
    const int s_lo = sp * per, s_hi = min(s_lo + per, kv_len);
    const bool has_new = FUSED && pos >= s_lo && pos < s_hi;  // this split holds the new token
    const int64_t kv_base = ((int64_t)b * a.HKV + j) * a.S * D;
    const int64_t mrow = (int64_t)b * a.ld_mask;

    // The wave's first block goes out before the prologue's arithmetic --
    // except the block that holds the new token, which its wave loads after
    // the workgroup has written that token's key and value (the barrier at
    // the end of the prologue orders the workgroup's own stores before its
    // loads).
    Blk cur;
    int s0 = s_lo + wave * kBlk;
    const bool first_new = has_new && pos >= s0 && pos < s0 + kBlk;
    if (!first_new && s0 < s_hi) load_block<DL, F32C>(a, kv_base, s0, s_hi, mrow, lane, cur);

    if constexpr (FUSED) {
        // raw rows: [0, G) query heads, G: key head j, G + 1: value head j;
        // each wave's 64 elements of one i share a row
        float* raw = &st_acc[0][0][0];
        for (int i = 0; i < NI; ++i) {
            const int e = tid + i * kAttnThreads;
            if (e / D < nrows) {
                const float v = bf16_to_f32((uint16_t)pre[i]);
                raw[e] = v;
                const float ss = wave_sum64(v * v);
                if (lane == 0) css[e >> 6] = ss;
            }
        }
        __syncthreads();
        // inverse RMS of each normed row (q heads and the key head), chunk
        // partials summed in column order
        if (tid <= G) {
            float ss = 0.0f;
            for (int q = 0; q < DL; ++q) ss += css[tid * DL + q];
            rinv[tid] = a.qn ? 1.0f / sqrtf(ss / (float)D + a.eps) : 1.0f;
        }
        __syncthreads();
        const int nout = G + (has_new ? 1 : 0);
        for (int i = 0; i < NI; ++i) {
            const int e = tid + i * kAttnThreads;
            const int r = e / D, d = e - r * D;
            if (r >= nout) continue;
            const int c = NC == 2 ? (i & 1) : 0;
            const int dp = d < D / 2 ? d + D / 2 : d - D / 2;
            float v = raw[r * D + d], rr = raw[r * D + dp];
            if (a.qn) {
                const float inv = rinv[r];
                const bool isq = r < G;  // selects, not a run-time index into a register array
                v = v * inv * bf16_to_f32((uint16_t)(isq ? nw_r[c][0] : nw_r[c][2]));
                rr = rr * inv * bf16_to_f32((uint16_t)(isq ? nw_r[c][1] : nw_r[c][3]));
            }
            if (d < D / 2) rr = -rr;
            const float o = v * raw_f32(cs_r[c], cs_kind) + rr * raw_f32(sn_r[c], cs_kind);
            if (r < G) {
                qf[r][d] = o;
            } else {  // the new key into the cache
                st_any(a.kc, F32C, kv_base + pos * D + d, o);
            }
        }
        if (has_new) {
            for (int d = tid; d < D; d += kAttnThreads) st_any(a.vc, F32C, kv_base + pos * D + d, raw[(G + 1) * D + d]);
        }
        if (a.seq_len && b == 0 && j == 0 && sp == 0 && tid == 0) *a.seq_len = pos + 1;
    } else {
        float* qflat = &qf[0][0];
        for (int i = 0; i < NI; ++i) {
            const int e = tid + i * kAttnThreads;
            if (e < G * D) qflat[e] = __uint_as_float(pre[i]);
        }
    }
    __syncthreads();

    if (first_new && s0 < s_hi) load_block<DL, F32C>(a, kv_base, s0, s_hi, mrow, lane, cur);

    // A operand: row `col` = query head j*G + col (zero rows from G on);
    // element e of step t is scale * q[32t + 8 grp + e], as bf16 hi + lo.
    // The operands are the same for every wave: built once into LDS (wave w
    // builds steps w, w + 4, ...) and read back per block.
    {
        const bool qv = col < G;
        const float sc = qv ? a.scale : 0.0f;
        const float* qrow = qf[qv ? col : 0];
        for (int t = wave; t < T; t += kAttnWaves) {
            float v[8];
            for (int e = 0; e < 8; ++e) v[e] = qrow[32 * t + 8 * grp + e] * sc;
            split8(v, qop[t][0][lane], qop[t][1][lane]);
        }
    }
    __syncthreads();

    // Score state: lane holds heads 4 grp + r (r < 4) at position col; m is
    // uniform over the 16 lanes of a group, l is this lane's share.
    float m[4], l[4];
    for (int r = 0; r < 4; ++r) {
        m[r] = kNegBig;
        l[r] = 0.0f;
    }
    float acc[GM][DL];  // VALU p v: head h, this lane's DL columns
    for (int h = 0; h < GM; ++h)
        for (int e = 0; e < DL; ++e) acc[h][e] = 0.0f;

    // One block: scores on the matrix cores, online softmax, p v on the VALU.
    auto process = [&](Blk& blk, const int s0) __attribute__((always_inline)) {
        const int kpos = s0 + col;
        const bool valid = kpos < s_hi;
        f32x4_t sc = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int t = 0; t < T; ++t) {
            const u32x4 qh = qop[t][0][lane], ql = qop[t][1][lane];
            sc = mfma16(qh, blk.kh[t], sc);
            sc = mfma16(ql, blk.kh[t], sc);
            if constexpr (F32C) sc = mfma16(qh, blk.kl[t], sc);
        }
        float alpha[4];
        const float mk = valid ? raw_f32(blk.mraw, a.mask_dtype) : 0.0f;
        for (int r = 0; r < 4; ++r) {
            const float s = valid ? sc[r] + mk : kNegBig;
            const float mn = fmaxf(m[r], max16(s));
            alpha[r] = fexp2((m[r] - mn) * kLog2e);
            const float pr = valid ? fexp2((s - mn) * kLog2e) : 0.0f;
            l[r] = l[r] * alpha[r] + pr;
            m[r] = mn;
            // every head slot of the block is written (rows past G hold
            // finite values of zero query rows and are never output)
            if (4 * grp + r < GM) p_lds[wave][col * GM + 4 * grp + r] = pr;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // rescale by head h's alpha (lane 16 (h / 4), element h % 4)
        for (int h = 0; h < GM; ++h) {
            const float al = bcast(alpha[h & 3], 16 * (h >> 2));
            for (int e = 0; e < DL; ++e) acc[h][e] *= al;
        }
        for (int p = 0; p < kBlk; ++p) {
            float vv[DL];
            for (int e = 0; e < DL; ++e) vv[e] = vword<DL, F32C>(blk.v[p], e);
            float pw[GM];
            for (int h = 0; h < GM; h += 4) {
                const float4 t = *reinterpret_cast<const float4*>(&p_lds[wave][p * GM + h]);
                pw[h] = t.x;
                pw[h + 1] = t.y;
                pw[h + 2] = t.z;
                pw[h + 3] = t.w;
            }
            for (int h = 0; h < GM; ++h)
                for (int e = 0; e < DL; ++e) acc[h][e] += pw[h] * vv[e];
        }
        // p_lds is rewritten by this wave's next block
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    constexpr int kStride = kAttnWaves * kBlk;
    for (; s0 < s_hi; s0 += kStride) {
        process(cur, s0);
        if (s0 + kStride < s_hi) load_block<DL, F32C>(a, kv_base, s0 + kStride, s_hi, mrow, lane, cur);
    }

    // Per-wave state to LDS: head 4 grp + r's m and l (l summed over the
    // group's 16 positions).
    __syncthreads();  // the prologue's raw rows share st_acc
    for (int r = 0; r < 4; ++r) {
        const float ls = sum16(l[r]);
        const int h = 4 * grp + r;
        if (col == 0 && h < G) {
            st_m[wave][h] = m[r];
            st_l[wave][h] = ls;
        }
    }
    for (int h = 0; h < GM; ++h)
        if (h < G)
            for (int e = 0; e < DL; ++e) st_acc[wave][h][DL * lane + e] = acc[h][e];
    __syncthreads();

    merge_and_combine<D, GM, kAttnWaves, D>(a, b, j, sp, nsp, kAttnWaves, tid, &st_m[0][0], &st_l[0][0],
                                            &st_acc[0][0][0], &last);
}

// Waves per workgroup of attn_bf16: eight, or four where 16 heads of 256 columns
// fill the LDS.
template <int DL, int GM, bool FUSED>
static void launch_attn(const AttnParams& a, bool f32c, dim3 grid, hipStream_t st) {
    const void* rows = FUSED ? static_cast<const void*>(a.qkv) : static_cast<const void*>(a.q);
    const int ld = (int)a.ld_qkv;  // bz_attn_step: checked to fit 32 bits
    if (f32c) {
        hipLaunchKernelGGL((attn_kernel<DL, GM, true, FUSED>), grid, dim3(64 * kAttnWaves), 0, st, rows, a.cosp, a.sinp,
                           a.pos, a.kc, a.vc, ld, a.G, a);
    } else if constexpr (DL <= 4) {
        constexpr int NWV = GM == 16 && DL == 4 ? 4 : 8;
        // G, HKV, whether cos / sin are fp32 and whether one row serves all:
        // what the first loads need in one preloaded word (grid.y <= 65535)
        const uint32_t shape =
            (uint32_t)a.G | (uint32_t)a.HKV << 5 | (a.cs_f32 ? 1u << 21 : 0u) | (a.ld_cs == 0 ? 1u << 22 : 0u);
        // no more splits than the longest context of this cache uses: a
        // workgroup without one still loads its prologue's rows before it knows
        // (MI355X, S = 1024, 41 positions, 16 / 8 heads of 128, 8 splits asked for:
        // 200 (row, kv head) pairs 7.89 -> 6.05 us, 512 16.6 -> 10.3, 96 5.42 -> 5.39;
        // 200 pairs over S = 2048, 16 splits 9.65 -> 4.99)
        if (a.S <= attn_unsplit(DL))
            grid.z = 1;
        else
            grid.z = std::min(a.split_cap, ((a.S + kBlk - 1) / kBlk + NWV - 1) / NWV);
        hipLaunchKernelGGL((attn_bf16<DL, GM, FUSED, NWV>), grid, dim3(64 * NWV), 0, st, rows, a.cosp, a.sinp, a.pos,
                           a.kc, a.vc, ld, shape, a);
    } else {
        hipLaunchKernelGGL((attn_kernel<DL, GM, false, FUSED>), grid, dim3(64 * kAttnWaves), 0, st, rows, a.cosp, a.sinp,
                           a.pos, a.kc, a.vc, ld, a.G, a);
    }
}

template <bool FUSED>
static int launch_attn_any(const AttnParams& a, int D, bool f32c, dim3 grid, hipStream_t st) {
    const bool g4 = a.G <= 4;
    switch (D) {
        case 64: g4 ? launch_attn<1, 4, FUSED>(a, f32c, grid, st) : launch_attn<1, 16, FUSED>(a, f32c, grid, st); break;
        case 128: g4 ? launch_attn<2, 4, FUSED>(a, f32c, grid, st) : launch_attn<2, 16, FUSED>(a, f32c, grid, st); break;
        case 256: g4 ? launch_attn<4, 4, FUSED>(a, f32c, grid, st) : launch_attn<4, 16, FUSED>(a, f32c, grid, st); break;
        default: launch_attn<8, 4, FUSED>(a, f32c, grid, st); break;
    }
    return hipGetLastError() == hipSuccess ? BZ_OK : BZ_ERR_LAUNCH;
}

static bool aligned(const void* p, uintptr_t n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; }

static size_t partial_floats(int B, int HQ, int D, int split) { return (size_t)B * HQ * split * (D + 4); }

// Checks shared by bz_attn_decode and bz_attn_step; fills the attention part
// of the parameters.
static int attn_setup(AttnParams& a, const void* k_cache, const void* v_cache, int cache_dtype, int B, int HQ, int HKV,
                      int D, int S, const void* mask, int mask_dtype, int64_t ld_mask, const int64_t* pos, float scale,
                      int split, void* workspace, void* out, int64_t ld_out) {
    if (!k_cache || !v_cache || !mask || !pos || !out) return BZ_ERR_INVALID_ARG;
    if (B < 1 || HQ < 1 || HKV < 1 || S < 1 || HQ % HKV) return BZ_ERR_INVALID_ARG;
    if (cache_dtype != BZ_DT_BF16 && cache_dtype != BZ_DT_F32) return BZ_ERR_INVALID_ARG;
    if (mask_dtype != BZ_DT_BF16 && mask_dtype != BZ_DT_F32 && mask_dtype != BZ_MASK_BOOL) return BZ_ERR_INVALID_ARG;
    if (split < 1 || split > BZ_ATTN_MAX_SPLIT || (split > 1 && !workspace)) return BZ_ERR_INVALID_ARG;
    if ((ld_mask != 0 && ld_mask < S) || ld_mask < 0 || ld_out < (int64_t)HQ * D) return BZ_ERR_SHAPE;
    const int G = HQ / HKV;
    if (D != 64 && D != 128 && D != 256 && D != 512) return BZ_ERR_UNSUPPORTED;
    if ((int64_t)S * D * 4 >= (int64_t(1) << 32)) return BZ_ERR_UNSUPPORTED;  // 32-bit offsets in one head's cache
    if (G > 16 || (G > 4 && D == 512)) return BZ_ERR_UNSUPPORTED;
    if (!aligned(k_cache, 16) || !aligned(v_cache, 16) || !aligned(out, 2) || !aligned(workspace, 4))
        return BZ_ERR_ALIGNMENT;
    a.kc = const_cast<void*>(k_cache);
    a.vc = const_cast<void*>(v_cache);
    a.mask = mask;
    a.ld_mask = ld_mask;
    a.mask_dtype = mask_dtype;
    a.pos = pos;
    a.scale = scale;
    a.HQ = HQ;
    a.HKV = HKV;
    a.G = G;
    a.S = S;
    a.split = split;
    a.split_cap = std::max(1, std::min<int>(split, (int)(256 / ((int64_t)B * HKV))));
    a.part = static_cast<float*>(workspace);
    a.counters = split > 1 ? reinterpret_cast<unsigned*>(a.part + partial_floats(B, HQ, D, split)) : nullptr;
    a.out = static_cast<uint16_t*>(out);
    a.ld_out = ld_out;
    return BZ_OK;
}

}  // namespace bz

using namespace bz;

extern "C" int bz_qkv_rope_cache(const void* qkv, int64_t ld_qkv, int32_t B, int32_t HQ, int32_t HKV, int32_t D,
                                 const void* q_norm, const void* k_norm, float eps, const void* cos, const void* sin,
                                 int32_t cs_dtype, int64_t ld_cs, const int64_t* pos, float* q_out, void* k_cache,
                                 void* v_cache, int32_t S, int32_t cache_dtype, int64_t* seq_len, void* stream) {
    if (!qkv || !cos || !sin || !pos || !q_out || !k_cache || !v_cache) return BZ_ERR_INVALID_ARG;
    if (B < 1 || HQ < 1 || HKV < 1 || S < 1 || (q_norm == nullptr) != (k_norm == nullptr)) return BZ_ERR_INVALID_ARG;
    if ((cs_dtype != BZ_DT_BF16 && cs_dtype != BZ_DT_F32) || (cache_dtype != BZ_DT_BF16 && cache_dtype != BZ_DT_F32))
        return BZ_ERR_INVALID_ARG;
    if (D < 2 || D % 2 || D > kMaxRopeDim || ld_qkv < (int64_t)(HQ + 2 * HKV) * D || ld_cs < 0) return BZ_ERR_SHAPE;
    hipLaunchKernelGGL(qkv_rope_cache_kernel, dim3(B, HQ + HKV), dim3(kRopeThreads), 0,
                       static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(qkv), ld_qkv, HQ, HKV, D,
                       static_cast<const uint16_t*>(q_norm), static_cast<const uint16_t*>(k_norm), eps, cos, sin,
                       cs_dtype == BZ_DT_F32, ld_cs, pos, q_out, k_cache, v_cache, S, cache_dtype == BZ_DT_F32,
                       seq_len);
    return hipGetLastError() == hipSuccess ? BZ_OK : BZ_ERR_LAUNCH;
}

extern "C" int32_t bz_attn_default_split(int32_t S) {
    const int32_t s = (S + 127) / 128;  // about 128 positions per workgroup at a full cache
    return s < 1 ? 1 : (s > 32 ? 32 : s);
}

extern "C" size_t bz_attn_workspace(int32_t B, int32_t HQ, int32_t HKV, int32_t D, int32_t split) {
    if (B < 1 || HQ < 1 || HKV < 1 || D < 1 || split <= 1) return 0;
    return partial_floats(B, HQ, D, split) * sizeof(float) + (size_t)B * HKV * sizeof(unsigned);
}

extern "C" int bz_attn_decode(const float* q, const void* k_cache, const void* v_cache, int32_t cache_dtype, int32_t B,
                              int32_t HQ, int32_t HKV, int32_t D, int32_t S, const void* mask, int32_t mask_dtype,
                              int64_t ld_mask, const int64_t* pos, float scale, int32_t split, void* workspace,
                              void* out, int64_t ld_out, void* stream) {
    if (!q) return BZ_ERR_INVALID_ARG;
    AttnParams a = {};
    int rc = attn_setup(a, k_cache, v_cache, cache_dtype, B, HQ, HKV, D, S, mask, mask_dtype, ld_mask, pos, scale,
                        split, workspace, out, ld_out);
    if (rc != BZ_OK) return rc;
    if (!aligned(q, 16)) return BZ_ERR_ALIGNMENT;
    a.q = q;
    return launch_attn_any<false>(a, D, cache_dtype == BZ_DT_F32, dim3(B, HKV, split),
                                  static_cast<hipStream_t>(stream));
}

extern "C" int bz_attn_step(const void* qkv, int64_t ld_qkv, int32_t B, int32_t HQ, int32_t HKV, int32_t D,
                            const void* q_norm, const void* k_norm, float eps, const void* cos, const void* sin,
                            int32_t cs_dtype, int64_t ld_cs, const int64_t* pos, void* k_cache, void* v_cache,
                            int32_t S, int32_t cache_dtype, int64_t* seq_len, const void* mask, int32_t mask_dtype,
                            int64_t ld_mask, float scale, int32_t split, void* workspace, void* out, int64_t ld_out,
                            void* stream) {
    if (!qkv || !cos || !sin || (q_norm == nullptr) != (k_norm == nullptr)) return BZ_ERR_INVALID_ARG;
    if (cs_dtype != BZ_DT_BF16 && cs_dtype != BZ_DT_F32) return BZ_ERR_INVALID_ARG;
    AttnParams a = {};
    int rc = attn_setup(a, k_cache, v_cache, cache_dtype, B, HQ, HKV, D, S, mask, mask_dtype, ld_mask, pos, scale,
                        split, workspace, out, ld_out);
    if (rc != BZ_OK) return rc;
    if (ld_qkv < (int64_t)(HQ + 2 * HKV) * D || ld_cs < 0) return BZ_ERR_SHAPE;
    if (ld_qkv > 0x7FFFFFFF) return BZ_ERR_UNSUPPORTED;  // a preloaded 32-bit kernel argument
    a.qkv = static_cast<const uint16_t*>(qkv);
    a.ld_qkv = ld_qkv;
    a.qn = static_cast<const uint16_t*>(q_norm);
    a.kn = static_cast<const uint16_t*>(k_norm);
    a.eps = eps;
    a.cosp = cos;
    a.sinp = sin;
    a.cs_f32 = cs_dtype == BZ_DT_F32;
    a.ld_cs = ld_cs;
    a.seq_len = seq_len;
    return launch_attn_any<true>(a, D, cache_dtype == BZ_DT_F32, dim3(B, HKV, split),
                                 static_cast<hipStream_t>(stream));
}
