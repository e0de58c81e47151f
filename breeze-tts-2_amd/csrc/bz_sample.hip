// CFG + HF-order sampling of one token per row in one launch (gfx950).
//
// Replaces the depth decoder's per-codebook sampling sequence
// (models/cudagraph/depth_decoder_graph.py:487-558, _cfg_sample): the CFG
// combination uncond + g * (cond - uncond), the invalid-codec-token mask
// (models/logits_process.py:7-25), temperature, top-k over a fixed workspace,
// top-p, softmax, multinomial, and argmax for greedy rows -- about twenty
// torch kernels -- with one workgroup per sampled row:
//
//   1. combined logits of the row (and its greedy argmax, first index of the
//      maximum, as torch.argmax) into LDS, divided by the temperature;
//   2. the first k ranks of the row in order (k = top_k, or the whole
//      workspace for top_k <= 0; the workspace is <= 1024 wide), by unique
//      64-bit keys (scaled value, then ascending index): a histogram of the
//      values picks the buckets that hold them and each one's rank comes
//      from its own bucket; rows that do not suit it take a radix select and
//      a bitonic sort;
//   3. their softmax (one rank per thread), an inclusive scan of it, and the
//      top-p prefix: rank r stays when r == 0 or the cumulative probability
//      before it is <= top_p (the reference's shifted mask), so the kept set
//      is a prefix of ranks;
//   4. one uniform draw u in [0, 1) (Philox4x32-10, Salmon, Moraes, Dror and
//      Shaw, "Parallel random numbers: as easy as 1, 2, 3", SC 2011; key =
//      the 64-bit seed, read from device memory so a captured graph picks up
//      a new one; counter = (the row's call count, row)) and the first
//      kept rank whose cumulative weight exceeds u times the kept total;
//   5. the token (sampled, or the argmax when do_sample is 0) to the row and
//      its unconditional twin; the row's call count is advanced, so graph
//      replays draw fresh numbers;
//   6. bz_sample_next only: the token also to a column of the frame's tokens,
//      and its row of the embedding table to the next step's input (that
//      replaced a clamp, a copy, an offset add, a clamp and an index-select
//      launch of about 2.5 us each).
// A greedy row that reports no probabilities stops after step 1.
//
// The random stream is this library's own, not torch's: the sampled tokens
// follow the same distribution as the reference's, not the same sequence.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "bz_device.h"
#include "bz_gemv.h"
#include "bz_sample.h"

namespace bz {
namespace {

constexpr int kSampleThreads = 1024;
constexpr int kSampleWidth = 4096;  // padded row: the largest vocabulary
constexpr int kSampleMaxK = 1024;   // top-k workspace: one rank per thread

// Philox4x32-10 of the paper above: 10 rounds of the 4x32 round function with
// its published multipliers and Weyl key increments.
__device__ __forceinline__ void philox4x32_10(uint32_t (&c)[4], uint32_t k0, uint32_t k1) {
    constexpr uint32_t kM0 = 0xD2511F53u, kM1 = 0xCD9E8D57u, kW0 = 0x9E3779B9u, kW1 = 0xBB67AE85u;
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = (uint64_t)kM0 * c[0], p1 = (uint64_t)kM1 * c[2];
        const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c[1] ^ k0, n1 = (uint32_t)p1;
        const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c[3] ^ k1, n3 = (uint32_t)p0;
        c[0] = n0;
        c[1] = n1;
        c[2] = n2;
        c[3] = n3;
        k0 += kW0;
        k1 += kW1;
    }
}

struct SampleParams {
    const float* logits;
    int64_t ld;
    int B, half, V, codec, max_k;
    const float* guidance;
    const float* temperature;
    const int64_t* top_k;
    const float* top_p;
    const int64_t* do_sample;
    const uint64_t* seed;
    uint64_t* counters;
    int64_t* tokens;
    float* cfg_out;
    float* probs_out;
    int64_t* out_tokens;  // optional: [B] with stride out_ld
    int64_t out_ld;
    const uint8_t* table;  // optional: embedding rows of row_bytes
    int64_t table_rows, row_bytes, first_row;
    uint8_t* emb;          // [B] rows, emb_ld bytes apart
    int64_t emb_ld;
};

// Sort key of a row entry: the temperature-scaled value mapped to an
// unsigned order (larger float -> larger key) in the high word, the inverted
// index in the low word, so keys are unique and a larger key is a larger
// value, or the same value at a smaller index (the order of torch.argmax).
__device__ __forceinline__ uint64_t entry_key(float s, int v) {
    const uint32_t b = __float_as_uint(s);
    const uint32_t u = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
    return ((uint64_t)u << 32) | (uint32_t)(0xFFFFFFFFu - (uint32_t)v);
}
__device__ __forceinline__ float key_value(uint64_t key) {
    const uint32_t u = (uint32_t)(key >> 32);
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u);
}
__device__ __forceinline__ int key_index(uint64_t key) { return (int)(0xFFFFFFFFu - (uint32_t)key); }

__device__ __forceinline__ uint64_t shfl_xor64(uint64_t v, int m) {
    const uint32_t lo = __shfl_xor((uint32_t)v, m, 64), hi = __shfl_xor((uint32_t)(v >> 32), m, 64);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ float wave_scan_incl(float v, int lane) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const float t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}

constexpr int kPerThread = kSampleWidth / kSampleThreads;  // row entries a thread holds
constexpr int NW = kSampleThreads / 64;
constexpr int kBuckets = kSampleThreads;  // value buckets of the fast order, one per thread
constexpr int kBucketCap = 64;            // fullest bucket the fast order ranks by comparing
constexpr float kExpSpan = 110.0f;        // expf(-kExpSpan) is 0 in fp32
static_assert(NW == 16, "one 16-lane row holds a value of each wave");
constexpr int kCand = kSampleMaxK + kBucketCap;

// Bucket of a scaled value, 0 for the row's maximum: subtraction, product
// with scale >= 0 and truncation each keep the order, so a smaller bucket
// never holds a smaller value.
__device__ __forceinline__ int value_bucket(float s, float top, float scale) {
    return min((int)((top - s) * scale), kBuckets - 1);
}

// The row's token, by one whole wave: to the row and its twin, and what the
// next step reads of it; the row's call count advances.
__device__ __forceinline__ void put_token(const SampleParams& p, int r, int tok, uint64_t cnt, int lane) {
    tok = tok < 0 ? 0 : (tok >= p.V ? p.V - 1 : tok);
    const bool twin = p.B >= 2;
    if (lane == 0) {
        p.tokens[r] = tok;
        if (twin) p.tokens[p.half + r] = tok;
        p.counters[r] = cnt + 1;
        if (p.out_tokens) {
            p.out_tokens[r * p.out_ld] = tok;
            if (twin) p.out_tokens[(p.half + r) * p.out_ld] = tok;
        }
    }
    if (!p.table) return;
    const int64_t row = min<int64_t>(max<int64_t>(p.first_row + tok, 0), p.table_rows - 1);
    const uint8_t* src = p.table + row * p.row_bytes;
    uint8_t* d0 = p.emb + r * p.emb_ld;
    uint8_t* d1 = p.emb + (p.half + r) * p.emb_ld;
    for (int64_t o0 = lane * 16; o0 < p.row_bytes; o0 += 4096) {  // four loads in flight: 4 KiB a turn
        u32x4 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = ldg16(src + min<int64_t>(o0 + 1024 * i, p.row_bytes - 16));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t o = o0 + 1024 * i;
            if (o < p.row_bytes) {
                *reinterpret_cast<u32x4*>(d0 + o) = v[i];
                if (twin) *reinterpret_cast<u32x4*>(d1 + o) = v[i];
            }
        }
    }
}

// Reductions over 16-lane rows and the wave in DPP moves: a step is one VALU
// operation where a shuffle is an LDS round trip.
template <int CTRL>
__device__ __forceinline__ int dpp_i32(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}
__device__ __forceinline__ int min16_dpp(int v) {
    v = min(v, dpp_i32<kDppXor1>(v));
    v = min(v, dpp_i32<kDppXor2>(v));
    v = min(v, dpp_i32<kDppHalfMirror>(v));
    return min(v, dpp_i32<kDppRowMirror>(v));
}
__device__ __forceinline__ float lane_f32(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ float wave_max_dpp(float v) {
    v = max16_dpp(v);
    return fmaxf(fmaxf(lane_f32(v, 0), lane_f32(v, 16)), fmaxf(lane_f32(v, 32), lane_f32(v, 48)));
}
__device__ __forceinline__ int wave_min_dpp(int v) {
    v = min16_dpp(v);
    return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}
// inclusive scan of each 16-lane row (row_shr 1, 2, 4, 8), then of the wave
__device__ __forceinline__ int row_scan_dpp(int v) {
    v += dpp_i32<0x111>(v);
    v += dpp_i32<0x112>(v);
    v += dpp_i32<0x114>(v);
    return v + dpp_i32<0x118>(v);
}
__device__ __forceinline__ int wave_scan_dpp(int v) {
    v = row_scan_dpp(v);
    v += __builtin_amdgcn_update_dpp(0, v, kDppRowBcast15, 0xA, 0xF, false);
    return v + __builtin_amdgcn_update_dpp(0, v, kDppRowBcast31, 0xC, 0xF, false);
}

struct SampleShared {
    uint64_t cand[kCand];          // the candidates, bucket by bucket
    uint64_t sorted[kSampleMaxK];  // the keys of ranks 0, 1, ...
    unsigned hist[kBuckets];       // counts, then where each bucket ends in cand
    float wsum[NW], wtop[NW], wlow[NW], wbest_v[NW];
    int wbest_i[NW];
    int wcount[NW];
    int ncand, sel_digit, sel_need, sel_count, pick, last_kept, nsel, full;
};

// The largest kk keys of the row in sh.sorted, descending, by a radix select
// over 8-bit digits and a bitonic sort: any keys, any ties.
__device__ __forceinline__ void select_general(SampleShared& sh, const uint64_t (&key)[kPerThread], int kk) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint64_t prefix = 0, mask = 0;
    int need = kk;
    if (tid == 0) sh.ncand = 0;
    for (int shift = 56; shift >= 0; shift -= 8) {
        if (tid < 256) sh.hist[tid] = 0u;
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kPerThread; ++q)
            if (key[q] != 0 && (key[q] & mask) == prefix) atomicAdd(&sh.hist[(key[q] >> shift) & 255u], 1u);
        __syncthreads();
        if (wave == 0) {
            // lane l covers digits 255 - 4l .. 252 - 4l (top down)
            unsigned c4[4], sum = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                c4[q] = sh.hist[255 - 4 * lane - q];
                sum += c4[q];
            }
            unsigned incl = sum;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const unsigned t = __shfl_up(incl, o, 64);
                if (lane >= o) incl += t;
            }
            unsigned above = incl - sum;  // keys in higher digits than this lane's
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (above < (unsigned)need && above + c4[q] >= (unsigned)need) {
                    sh.sel_digit = 255 - 4 * lane - q;
                    sh.sel_need = need - (int)above;
                    sh.sel_count = (int)c4[q];
                }
                above += c4[q];
            }
        }
        __syncthreads();
        prefix |= (uint64_t)sh.sel_digit << shift;
        mask |= (uint64_t)255u << shift;
        need = sh.sel_need;
        if (sh.sel_count == need) break;  // workgroup-uniform
    }
    // the kk selected keys, padded with zeros to P (a power of two >= 64),
    // then a bitonic sort, descending: partners less than 64 apart trade
    // through wave shuffles, wider ones through LDS
    const int P = max(64, 1 << (32 - __clz(kk - 1)));
#pragma unroll
    for (int q = 0; q < kPerThread; ++q)
        if (key[q] != 0 && key[q] >= prefix) sh.cand[atomicAdd(&sh.ncand, 1)] = key[q];
    __syncthreads();
    uint64_t mine = tid < kk ? sh.cand[tid] : 0;
    for (int lk = 1; (1 << lk) <= P; ++lk) {
        const int k = 1 << lk;
        for (int lj = lk - 1; lj >= 0; --lj) {
            const int j = 1 << lj;
            uint64_t theirs;
            if (j < 64) {
                theirs = shfl_xor64(mine, j);
            } else {
                __syncthreads();
                if (tid < P) sh.cand[tid] = mine;
                __syncthreads();
                theirs = tid < P ? sh.cand[tid ^ j] : 0;
            }
            const bool lower = (tid & j) == 0, desc = (tid & k) == 0;
            const uint64_t hi = mine > theirs ? mine : theirs, lo = mine > theirs ? theirs : mine;
            if (tid < P) mine = (lower == desc) ? hi : lo;
        }
    }
    sh.sorted[tid] = mine;
    __syncthreads();
}

// One workgroup a row, so latency is all of it: parameters and logits are
// requested together, reductions stay in DPP moves, and the chain of barriers
// and LDS round trips is short.  Measured on MI355X in a graph of 16 launches,
// V = 2051, B = 2, with probs_out: 14.6 us a launch with the radix select and
// shuffle reductions for every row, 6.0 us now (top_k = 50); 20.8 and 7.9 us
// at top_k = 1000.
__global__ void __launch_bounds__(kSampleThreads) sample_cfg_kernel(SampleParams p) {
    __shared__ SampleShared sh;
    const int r = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const float* cond = p.logits + (int64_t)r * p.ld;
    const float* uncond = p.logits + (int64_t)(p.B >= 2 ? p.half + r : r) * p.ld;
    const float g = p.B >= 2 ? p.guidance[r] : 0.0f;
    const float temp = p.temperature[r];
    const int64_t tk = p.top_k[r];
    const float top_p = p.top_p[r];
    const bool sample = p.do_sample[r] != 0;
    const uint64_t cnt = p.counters[r], seed = *p.seed;
    float* pr = p.probs_out ? p.probs_out + (int64_t)r * p.V : nullptr;

    // 1. combined logits, greedy argmax, the scaled entries' keys (registers)
    float best_v = -INFINITY, top = -INFINITY, low = INFINITY;
    int best_i = 0x7FFFFFFF;
    float sv[kPerThread], cv[kPerThread], uv[kPerThread];
#pragma unroll
    for (int q = 0; q < kPerThread; ++q) {  // every load is in flight before the first is used
        const int v = min(tid + q * kSampleThreads, p.V - 1);
        cv[q] = cond[v];
        uv[q] = uncond[v];
    }
    sh.hist[tid] = 0u;
    uint64_t key[kPerThread];
#pragma unroll
    for (int q = 0; q < kPerThread; ++q) {
        const int v = tid + q * kSampleThreads;
        key[q] = 0;  // absent (below every entry's key)
        sv[q] = -INFINITY;
        if (v < p.V) {
            float c = cv[q];
            if (p.B >= 2) c = uv[q] + g * (c - uv[q]);
            if (v >= p.codec) c = -INFINITY;
            if (p.cfg_out) p.cfg_out[(int64_t)r * p.V + v] = c;
            if (pr) pr[v] = 0.0f;  // (barriers lie between this and step 3)
            if (c > best_v || best_i == 0x7FFFFFFF) {  // ascending v: the first maximum wins
                best_v = c;
                best_i = v;
            }
            sv[q] = c / temp;
            key[q] = entry_key(sv[q], v);
            // a NaN counts as infinite: neither is left to the fast order
            top = sv[q] <= top ? top : (sv[q] > top ? sv[q] : INFINITY);
            if (sv[q] > -INFINITY) low = fminf(low, sv[q]);
        }
    }
    top = wave_max_dpp(top);
    low = -wave_max_dpp(-low);
    if (top < INFINITY) {  // no NaNs: the maximum, then its first index
        const float bv = wave_max_dpp(best_v);
        best_i = wave_min_dpp(best_v == bv ? best_i : 0x7FFFFFFF);
        best_v = bv;
    } else {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const float ov = __shfl_xor(best_v, o, 64);
            const int oi = __shfl_xor(best_i, o, 64);
            if (ov > best_v || (ov == best_v && oi < best_i)) {
                best_v = ov;
                best_i = oi;
            }
        }
    }
    if (lane == 0) {
        sh.wbest_v[wave] = best_v;
        sh.wbest_i[wave] = best_i;
        sh.wtop[wave] = top;
        sh.wlow[wave] = low;
    }
    if (tid == 0) {
        sh.nsel = kSampleWidth;
        sh.full = 0;
        sh.pick = 0x7FFFFFFF;
        sh.last_kept = 0;
    }
    __syncthreads();
    top = lane_f32(max16_dpp(sh.wtop[lane & 15]), 0);
    low = -lane_f32(max16_dpp(-sh.wlow[lane & 15]), 0);
    int greedy;
    if (top < INFINITY) {
        best_v = sh.wbest_v[lane & 15];
        best_i = sh.wbest_i[lane & 15];
        greedy = __builtin_amdgcn_readlane(min16_dpp(best_v == max16_dpp(best_v) ? best_i : 0x7FFFFFFF), 0);
    } else {
        float bv = sh.wbest_v[0];
        greedy = sh.wbest_i[0];
        for (int w = 1; w < NW; ++w) {
            const float ov = sh.wbest_v[w];
            const int oi = sh.wbest_i[w];
            if (ov > bv || (ov == bv && oi < greedy)) {
                bv = ov;
                greedy = oi;
            }
        }
    }

    // A greedy row with no probabilities to report needs only the argmax:
    // skip the order, softmax and draw; the call count advances all the same.
    if (!sample && !p.probs_out) {
        if (wave == 0) put_token(p, r, greedy, cnt, lane);
        return;
    }

    // 2. the entries of ranks 0 .. kk - 1 in order (kk = top_k, or the whole
    //    workspace).  Fast order: a histogram of the values over kBuckets
    //    equal steps from the maximum down, the candidates (the buckets that
    //    hold the first kk entries, whole) grouped by bucket, and each one's
    //    rank from the few others of its bucket.  Entries more than kExpSpan
    //    below the maximum weigh 0, as -inf does, and take no rank.  Rows
    //    with infinities or NaNs, and rows crowded into a bucket, take the
    //    radix select instead.
    const int kk = tk > 0 ? (int)min<int64_t>(tk, p.max_k) : p.max_k;
    low = fmaxf(low, top - kExpSpan);
    const float range = top - low;
    bool fast = top < INFINITY && top > -INFINITY;  // (then low and range are finite)
    int nrank = kk;                                 // ranks in sh.sorted
    if (fast) {                                     // workgroup-uniform
        const float scale = range > 1e-30f ? (float)kBuckets / range : 0.0f;
#pragma unroll
        for (int q = 0; q < kPerThread; ++q)
            if (sv[q] >= low) atomicAdd(&sh.hist[value_bucket(sv[q], top, scale)], 1u);
        __syncthreads();
        const int c = (int)sh.hist[tid];
        int incl = wave_scan_dpp(c);
        if (lane == 63) sh.wcount[wave] = incl;
        __syncthreads();
        const int upto = row_scan_dpp(sh.wcount[lane & 15]);  // entries of waves 0 .. lane & 15
        if (wave) incl += __builtin_amdgcn_readlane(upto, wave - 1);
        nrank = min(kk, __builtin_amdgcn_readlane(upto, 15));
        const int start = incl - c;
        if (start < nrank && incl >= nrank) sh.nsel = incl;  // the last bucket taken
        if (c > kBucketCap && start < nrank) sh.full = 1;
        sh.hist[tid] = (unsigned)start;
        __syncthreads();
        fast = !sh.full;
        if (fast) {
            const int n = sh.nsel;  // < nrank + kBucketCap <= kCand
#pragma unroll
            for (int q = 0; q < kPerThread; ++q)
                if (sv[q] >= low) {
                    const int b = value_bucket(sv[q], top, scale);
                    // buckets past the last taken start at n: entries that
                    // would go there add nothing
                    if (sh.hist[b] < (unsigned)n) sh.cand[atomicAdd(&sh.hist[b], 1u)] = key[q];
                }
            __syncthreads();
            for (int t = tid; t < n; t += kSampleThreads) {
                const uint64_t mine = sh.cand[t];
                const int b = value_bucket(key_value(mine), top, scale);
                const int lo = b ? (int)sh.hist[b - 1] : 0, hi = (int)sh.hist[b];
                int rank = lo;
                for (int j = lo; j < hi; j += 4) {  // four reads in flight
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint64_t other = sh.cand[min(j + i, kCand - 1)];
                        rank += j + i < hi && other > mine;
                    }
                }
                if (rank < nrank) sh.sorted[rank] = mine;
            }
            __syncthreads();
        }
    }
    if (!fast) {
        nrank = kk;
        select_general(sh, key, kk);
    }

    // 3. thread t = rank t: top-k softmax weights, scan, top-p prefix, draw.
    //    The kept set is a prefix of ranks: rank 0, and the ranks whose
    //    cumulative probability before them is <= top_p.
    if (nrank <= 64 && wave) return;  // wave 0 holds every rank: no more barriers
    const float m_s = key_value(sh.sorted[0]);
    const uint64_t mine = tid < nrank ? sh.sorted[tid] : 0;
    const float sv_t = key_value(mine);
    const int si_t = key_index(mine);
    const float e = (tid < nrank && sv_t > -INFINITY) ? expf(sv_t - m_s) : 0.0f;
    uint32_t c[4] = {(uint32_t)cnt, (uint32_t)(cnt >> 32), (uint32_t)r, 0u};
    philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
    const float u = (float)(c[0] >> 8) * (1.0f / 16777216.0f);
    float inc = wave_scan_incl(e, lane);
    if (nrank <= 64) {
        const float total = __shfl(inc, 63, 64);
        const bool kept = e > 0.0f && (tid == 0 || (inc - e) / total <= top_p);
        const float ke = kept ? e : 0.0f;
        float kept_total = ke;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) kept_total += __shfl_xor(kept_total, o, 64);
        if (pr && kept) pr[si_t] = ke / kept_total;
        const uint64_t over = __ballot(kept && inc > u * kept_total), any = __ballot(kept);
        // the first kept rank past the draw; rounding at the top end: the last kept one
        const int at = over ? __ffsll((unsigned long long)over) - 1
                            : (any ? 63 - __clzll((long long)any) : 0);
        put_token(p, r, sample ? __builtin_amdgcn_readlane(si_t, at) : greedy, cnt, lane);
        return;
    }
    if (lane == 63) sh.wsum[wave] = inc;
    __syncthreads();
    float before_w = 0.0f, total = 0.0f;
    for (int w = 0; w < NW; ++w) {
        if (w < wave) before_w += sh.wsum[w];
        total += sh.wsum[w];
    }
    inc += before_w;
    const float exc = inc - e;
    const bool kept = e > 0.0f && (tid == 0 || exc / total <= top_p);
    __syncthreads();  // wsum is reused below
    const float ke = kept ? e : 0.0f;
    float ks = ke;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ks += __shfl_xor(ks, o, 64);
    if (lane == 0) sh.wsum[wave] = ks;
    __syncthreads();
    float kept_total = 0.0f;
    for (int w = 0; w < NW; ++w) kept_total += sh.wsum[w];
    if (pr && kept) pr[si_t] = ke / kept_total;
    const uint64_t over = __ballot(kept && inc > u * kept_total), any = __ballot(kept);
    if (lane == 0) {  // one LDS atomic a wave
        if (any) atomicMax(&sh.last_kept, tid + 63 - __clzll((long long)any));
        if (over) atomicMin(&sh.pick, tid + __ffsll((unsigned long long)over) - 1);
    }
    __syncthreads();
    if (wave == 0) {
        const int at = sh.pick == 0x7FFFFFFF ? sh.last_kept : sh.pick;
        put_token(p, r, sample ? key_index(sh.sorted[at]) : greedy, cnt, lane);
    }
}

}  // namespace
}  // namespace bz

using namespace bz;

static int fill_params(SampleParams& p, const float* logits, int64_t ld_logits, int32_t B, int32_t V, int32_t codec_size,
                       int32_t max_k, const float* guidance, const float* temperature, const int64_t* top_k,
                       const float* top_p, const int64_t* do_sample, const uint64_t* seed, uint64_t* counters,
                       int64_t* tokens, float* cfg_out, float* probs_out) {
    if (!logits || !temperature || !top_k || !top_p || !do_sample || !seed || !counters || !tokens)
        return BZ_ERR_INVALID_ARG;
    if (B < 1 || (B > 1 && B % 2) || V < 1 || V > kSampleWidth || ld_logits < V) return BZ_ERR_INVALID_ARG;
    if (codec_size < 1 || codec_size > V || max_k < 1 || max_k > kSampleMaxK || max_k > V) return BZ_ERR_INVALID_ARG;
    if (B >= 2 && !guidance) return BZ_ERR_INVALID_ARG;
    p = SampleParams{};
    p.logits = logits;
    p.ld = ld_logits;
    p.B = B;
    p.half = B == 1 ? 1 : B / 2;
    p.V = V;
    p.codec = codec_size;
    p.max_k = max_k;
    p.guidance = guidance;
    p.temperature = temperature;
    p.top_k = top_k;
    p.top_p = top_p;
    p.do_sample = do_sample;
    p.seed = seed;
    p.counters = counters;
    p.tokens = tokens;
    p.cfg_out = cfg_out;
    p.probs_out = probs_out;
    return BZ_OK;
}

static int launch(const SampleParams& p, void* stream) {
    hipLaunchKernelGGL(sample_cfg_kernel, dim3(p.half), dim3(kSampleThreads), 0, static_cast<hipStream_t>(stream), p);
    return hipGetLastError() == hipSuccess ? BZ_OK : BZ_ERR_LAUNCH;
}

extern "C" int bz_sample_cfg(const float* logits, int64_t ld_logits, int32_t B, int32_t V, int32_t codec_size,
                             int32_t max_k, const float* guidance, const float* temperature, const int64_t* top_k,
                             const float* top_p, const int64_t* do_sample, const uint64_t* seed, uint64_t* counters,
                             int64_t* tokens, float* cfg_out, float* probs_out, void* stream) {
    SampleParams p;
    const int rc = fill_params(p, logits, ld_logits, B, V, codec_size, max_k, guidance, temperature, top_k, top_p,
                               do_sample, seed, counters, tokens, cfg_out, probs_out);
    return rc == BZ_OK ? launch(p, stream) : rc;
}

extern "C" int bz_sample_next(const float* logits, int64_t ld_logits, int32_t B, int32_t V, int32_t codec_size,
                              int32_t max_k, const float* guidance, const float* temperature, const int64_t* top_k,
                              const float* top_p, const int64_t* do_sample, const uint64_t* seed, uint64_t* counters,
                              int64_t* tokens, float* cfg_out, float* probs_out, int64_t* out_tokens, int64_t out_ld,
                              const void* table, int64_t table_rows, int64_t row_bytes, int64_t first_row, void* emb,
                              int64_t emb_ld, void* stream) {
    SampleParams p;
    const int rc = fill_params(p, logits, ld_logits, B, V, codec_size, max_k, guidance, temperature, top_k, top_p,
                               do_sample, seed, counters, tokens, cfg_out, probs_out);
    if (rc != BZ_OK) return rc;
    if (out_tokens && out_ld < 1) return BZ_ERR_INVALID_ARG;
    if (table) {
        if (!emb || table_rows < 1 || row_bytes < 16 || first_row < 0) return BZ_ERR_INVALID_ARG;
        if (row_bytes % 16 || emb_ld % 16 || emb_ld < row_bytes) return BZ_ERR_SHAPE;
        if ((reinterpret_cast<uintptr_t>(table) | reinterpret_cast<uintptr_t>(emb)) & 15) return BZ_ERR_ALIGNMENT;
    }
    p.out_tokens = out_tokens;
    p.out_ld = out_ld;
    p.table = static_cast<const uint8_t*>(table);
    p.table_rows = table_rows;
    p.row_bytes = row_bytes;
    p.first_row = first_row;
    p.emb = static_cast<uint8_t*>(emb);
    p.emb_ld = emb_ld;
    return launch(p, stream);
}
