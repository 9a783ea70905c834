// Token sampling on the device (gfx950): Sampler::sample
// (src/model/sampler.rs:133-196), bit-identical to the reference on the same
// logits, parameters and xorshift64 state, with two cases the reference
// leaves open: its top-k and top-p sorts are unstable, so equal values that
// straddle the cut may come in any order there (here: index order, equal to
// the reference whenever no such tie straddles the cut), and with NaN values
// their comparator is not an order at all, so the kept set is unspecified
// (here: an error, under top-k and top-p alike).
//
// The reference, on a copy of the logits:
//   repetition penalty (:151-164)   each distinct history id once:
//                                   l > 0 ? l / r : l * r
//   temperature (:166-176)          l *= 1 / t
//   top-k (:201-223)                l < (k-th largest) -> -inf
//   softmax_to_probs (:225-252)     max; e = exp(l - max); Σe left to right;
//                                   e *= 1 / Σ
//   top-p (:254-311)                descending order, running f32 sum until
//                                   it reaches p, the rest zeroed; Σ left to
//                                   right; p *= 1 / Σ
//   multinomial (:178-196)          total = Σp left to right; r = u * total;
//                                   the first i whose running sum reaches r
// Two routes, the same result bit for bit:
//  * top-k (0 < k < n, k <= kListCap): only the values at or above the k-th
//    largest have a non-zero probability, and a zero term changes none of the
//    running sums.
//    k_sample_scan (penalty, temperature, and a histogram of the values' top
//    12 key bits), k_sample_pick (the values from the k-th largest's bin up,
//    per workgroup in index order) and k_sample_topk (one workgroup: the k-th
//    largest, then softmax, top-p and the draw on the kept values in LDS).
//  * otherwise, or when more than kListCap values reach that bin: all n
//    values, the element-wise work over many workgroups and each
//    left-to-right sum by one (block_seq).  The descending orders come from a
//    stable device radix sort (rocPRIM) of order-preserving integer keys.
// Equal probabilities at the top-p cut are taken in index order; the
// reference's unstable sort leaves that order open.  exp is glibc's expf,
// restated in wm_expf.h.
#include <rocprim/device/device_radix_sort.hpp>

#include <cmath>
#include <cstdio>
#include <vector>

#include "wm_internal.h"
#include "wm_seqsum.h"
#include "wm_terms.h"

namespace {

constexpr int kSampleThreads = 1024;  // the one-workgroup kernels
constexpr int kScanThreads = 256;     // the kernels over many workgroups
constexpr uint32_t kStrip = 1024;     // values a k_sample_scan workgroup takes at a time
constexpr uint32_t kMaxParts = 1024;  // workgroups of those kernels
constexpr uint32_t kBins = 4096;      // histogram of the key's top 12 bits
constexpr uint32_t kListCap = 3840;   // values k_sample_topk holds in LDS
constexpr uint32_t kNewIds = 32;      // history ids passed as arguments

enum : uint32_t {
    SAMPLE_RUNNING = 0,
    SAMPLE_DONE = 1,         // id valid
    SAMPLE_NOT_POSITIVE = 2, // multinomial: total <= 0 or not finite (total valid)
    SAMPLE_NAN_ORDER = 3,    // NaN values to sort: top-k's logits, or top-p's probabilities
    SAMPLE_LIST_FULL = 4,    // top-k: more than kListCap values from the k-th largest's bin up
};

// The result, written to host memory by the kernel that ends the draw.
struct sample_result {
    uint32_t status;
    uint32_t id;
    float total;
};

// Between the kernels of one draw.  `nan` and the histogram are zero between
// draws: the last kernel to read them clears them.
struct sample_state {
    uint32_t nan;         // NaN among the values to sort
    uint32_t bin, above;  // top-k: the k-th largest's bin, the values above that bin
    float inv;            // 1 / Σexp (1 when Σ is not positive: unnormalised)
};

enum { TOPK_NONE = 0, TOPK_ALL = 1, TOPK_THRESHOLD = 2 };
enum { TOPP_NONE = 0, TOPP_ONE_HOT = 1, TOPP_CUT = 2, TOPP_KEEP_ALL = 3 };

struct sample_args {
    const float *logits;
    uint32_t n;
    uint32_t parts, per;  // workgroups of the wide kernels, values each (a multiple of kStrip)
    float *work, *probs;
    uint32_t *keys, *vals;          // sort inputs; k_sample_pick's lists
    const uint32_t *skeys, *svals;  // sort outputs
    uint32_t *hist;                 // [kBins]
    uint32_t *count;                // [parts] values each k_sample_pick workgroup listed
    float *pmax;                    // [parts] maxima
    sample_state *st;
    sample_result *out;  // host memory
    uint32_t *ids;       // the history on the device: n_ids entries, then n_new more
    uint32_t n_ids, n_new;
    uint32_t new_ids[kNewIds];
    int use_rep;
    float rep;
    int use_temp;
    float inv_t;
    int topk_mode;
    int list;  // top-k by list: the histogram is wanted
    uint32_t k;
    int topp_mode;
    float top_p;
    float unit;  // the xorshift64 draw in [0, 1)
};

// Order-preserving keys: key(a) < key(b) iff a < b for non-NaN floats
// (-0 below +0, which no phase distinguishes).
__device__ __forceinline__ uint32_t order_key(float v) {
    const uint32_t b = __float_as_uint(v);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float key_value(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}
constexpr uint32_t kKeyPosZero = 0x80000000u, kKeyNegZero = 0x7fffffffu;

// Sources of left-to-right sums: f(i) is term i, f.get8(i, n, v) terms
// i .. i+7 (wm::terms_get8).
struct plain_terms {
    const float *a;
    __device__ __forceinline__ float map(float x, uint32_t) const { return x; }
    __device__ __forceinline__ float operator()(uint32_t i) const { return a[i]; }
    __device__ __forceinline__ void get8(uint32_t i, uint32_t n, float (&v)[8]) const {
        wm::terms_get8(*this, a, i, n, v);
    }
};
// values held as order keys (the sorted probabilities)
struct key_terms {
    const uint32_t *k;
    __device__ __forceinline__ float map(float x, uint32_t) const { return key_value(__float_as_uint(x)); }
    __device__ __forceinline__ float operator()(uint32_t i) const { return key_value(k[i]); }
    __device__ __forceinline__ void get8(uint32_t i, uint32_t n, float (&v)[8]) const {
        wm::terms_get8(*this, reinterpret_cast<const float *>(k), i, n, v);
    }
};
// probabilities exp * inv after top-p (entries at or after the cut's last
// one, in the sorted order, are the kept ones) and its renormalisation
struct prob_terms {
    const float *e;
    float inv, inv2;
    bool cut;
    float cut_p;        // the last kept entry of the descending order
    uint32_t cut_i;
    __device__ __forceinline__ float map(float x, uint32_t i) const {
        const float p = x * inv;
        const bool keep = !cut || p > cut_p || (p == cut_p && i <= cut_i);
        return keep ? p * inv2 : 0.0f;
    }
    __device__ __forceinline__ float operator()(uint32_t i) const { return map(e[i], i); }
    __device__ __forceinline__ void get8(uint32_t i, uint32_t n, float (&v)[8]) const {
        wm::terms_get8(*this, e, i, n, v);
    }
};

// argmax as lm_head.rs:161-174 (`if v > best`, starting from a[0]): index 0
// when a[0] is NaN, else the first index of the maximum over the non-NaN
// values (a NaN never compares greater).  Every thread gets the result.
template <typename F>
__device__ uint32_t block_argmax_first(const F &a, uint32_t n, float *rv, uint32_t *ri) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    float bv = -INFINITY;
    uint32_t bi = 0xffffffffu;
    for (uint64_t i = tid; i < n; i += kSampleThreads) {  // (i passes 2^32 where n is close to it)
        const float v = a((uint32_t)i);
        if (!isnan(v) && (bi == 0xffffffffu || v > bv)) {
            bv = v;
            bi = (uint32_t)i;
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(bv, o, 64);
        const uint32_t oi = __shfl_xor(bi, o, 64);
        const bool take = oi != 0xffffffffu && (bi == 0xffffffffu || ov > bv || (ov == bv && oi < bi));
        bv = take ? ov : bv;
        bi = take ? oi : bi;
    }
    wm_sync_lds();
    if (lane == 0) {
        rv[wid] = bv;
        ri[wid] = bi;
    }
    wm_sync_lds();
    bv = rv[0];
    bi = ri[0];
    for (int w = 1; w < kSampleThreads / 64; w++) {
        const float ov = rv[w];
        const uint32_t oi = ri[w];
        if (oi != 0xffffffffu && (bi == 0xffffffffu || ov > bv || (ov == bv && oi < bi))) {
            bv = ov;
            bi = oi;
        }
    }
    return isnan(a(0)) || bi == 0xffffffffu ? 0u : bi;
}

// ---------------------------------------------------------------------------
// sums over an LDS list, by one wave (all 64 lanes, same result)
// ---------------------------------------------------------------------------

// Left-to-right sum of a[0..n), a[] >= 0 in LDS: up to 512 terms one by one
// (a lane holds a term, read as a scalar), longer lists by the one-wave
// algorithm.
__device__ float list_sum(const float *a, uint32_t n) {
    if (n > 512) return wm::seq_sum_nonneg(a, n);
    const uint32_t lane = threadIdx.x & 63;
    float s = 0.0f;
    for (uint32_t b = 0; b < n; b += 64) {
        const float x = b + lane < n ? a[b + lane] : 0.0f;
        const uint32_t m = min(64u, n - b);
        for (uint32_t l = 0; l < m; l += 8)  // zeros past the end change nothing
#pragma unroll
            for (uint32_t j = 0; j < 8; j++)
                s = s + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), (int)(l + j)));
    }
    return s;
}

// The first i in [0, n) at which the left-to-right sum a[0] + ... + a[i]
// reaches r (>= r), or n if it never does; the terms are non-negative and
// finite, so the running sum never decreases.
__device__ uint32_t list_first_reach(const float *a, uint32_t n, float r) {
    const uint32_t lane = threadIdx.x & 63;
    float s = 0.0f;
    for (uint32_t b = 0; b < n; b += 64) {
        const float x = b + lane < n ? a[b + lane] : 0.0f;
        const uint32_t m = min(64u, n - b);
        for (uint32_t l = 0; l < m; l += 8) {
            const float s0 = s;
#pragma unroll
            for (uint32_t j = 0; j < 8; j++)
                s = s + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), (int)(l + j)));
            if (s >= r) {
                s = s0;
                for (uint32_t j = 0; j < 8 && b + l + j < n; j++) {
                    s = s + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), (int)(l + j)));
                    if (s >= r) return b + l + j;
                }
                return n;
            }
        }
    }
    return n;
}

// ---------------------------------------------------------------------------
// sums over n values, by one 1024-thread workgroup
// ---------------------------------------------------------------------------
//
// The one-wave sum of wm_seqsum.h one level up.  Chunks of 512 terms: a
// float64 prefix over the chunk totals predicts the running sum's binade at
// each chunk, every wave forms chunks' integer increments Σ RN_int(a / ulp)
// for that binade (a halfway, huge or non-finite term marks the chunk), and
// one wave advances over runs of unmarked chunks with an integer prefix sum.
// A chunk that is marked, whose predicted binade is not the running sum's,
// or that would leave the binade is added by the one-wave algorithm from the
// exact sum before it, so the prediction is never trusted and every outcome
// is the left-to-right sum.  A chunk of zeros changes no sum.  128256 terms
// have about 15-25 chunks to add that way (the leading ones, where the sum
// doubles often, then halfway terms), whose serial adds bound it: about 50 us
// a sum, where one wave over all the terms took 250-300.  Draws without
// top-k, 128256 values, a call with its result on the host: 646 -> 166 us,
// with top-p 0.9 1022 -> 417 us.
constexpr uint32_t kChunks = 512;  // chunks per round
struct block_seq_lds {
    double tot[kChunks];    // chunk totals, then the prefix before each
    uint32_t inc[kChunks];  // increments (clamped to 2^24), kMarked, kZeros
    uint32_t ef[kChunks];   // predicted exponent field
    float pre[kChunks];     // exact sum before the chunk
    float s;
    uint32_t hit;
};
constexpr uint32_t kMarked = 0xffffffffu, kZeros = 0xfffffffeu;

// The left-to-right sum of f(0) .. f(n-1); with REACH, *hit is the first
// index whose running sum reaches r (n if none does) and the sum is that of
// the rounds up to it.  Every thread gets both.
template <bool REACH, typename F>
__device__ float block_seq(const F &f, uint32_t n, float r, uint32_t *hit, block_seq_lds &L) {
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wid = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    constexpr uint32_t kWaves = kSampleThreads / 64;
    float s = 0.0f;
    double carry = 0.0;
    for (uint64_t base = 0; base < n; base += (uint64_t)kChunks * wm::kSeqBatch) {
        const uint32_t b0 = (uint32_t)base;
        const uint32_t nch = (uint32_t)min((uint64_t)kChunks, (n - base + wm::kSeqBatch - 1) / wm::kSeqBatch);
        for (uint32_t c = wid; c < nch; c += kWaves) {
            float v[8];
            f.get8(b0 + c * wm::kSeqBatch + 8 * lane, n, v);
            double t = 0.0;
#pragma unroll
            for (int j = 0; j < 8; j++) t += (double)v[j];
            t = wm_wave_scan_f64(t);
            if (lane == 63) L.tot[c] = t;
        }
        __syncthreads();
        if (wid == 0) {  // prefixes: lane l takes chunks 8l .. 8l+7
            double t[8], own = 0.0;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                t[j] = 8 * lane + j < nch ? L.tot[8 * lane + j] : 0.0;
                own += t[j];
            }
            double p = carry + (wm_wave_scan_f64(own) - own);
#pragma unroll
            for (int j = 0; j < 8; j++) {
                L.tot[8 * lane + j] = p;
                p += t[j];
            }
            if (lane == 63) carry = p;
            carry = __longlong_as_double((long long)(((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)((unsigned long long)__double_as_longlong(carry) >> 32), 63) << 32) |
                                                     (unsigned)__builtin_amdgcn_readlane((int)(unsigned long long)__double_as_longlong(carry), 63)));
        }
        __syncthreads();
        for (uint32_t c = wid; c < nch; c += kWaves) {
            float v[8];
            f.get8(b0 + c * wm::kSeqBatch + 8 * lane, n, v);
            const uint32_t ef = __float_as_uint((float)L.tot[c]) >> 23;
            const int sh = 150 - (int)ef;
            uint32_t d = 0;
            bool bad = ef - 1u >= 254u, any = false;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float q = ldexpf(v[j], sh);
                const bool fin = q < 0x1p22f;
                const float qq = fin ? q : 0.0f;
                bad = bad || !fin || qq - floorf(qq) == 0.5f;
                any = any || !(v[j] == 0.0f);
                d += (uint32_t)rintf(qq);
            }
            d = (uint32_t)__builtin_amdgcn_readlane((int)wm::wave_scan_u32(min(d, 1u << 24)), 63);
            const bool wbad = __ballot(bad) != 0, wany = __ballot(any) != 0;
            if (lane == 0) {
                L.inc[c] = !wany ? kZeros : wbad ? kMarked : min(d, 1u << 24);
                L.ef[c] = ef;
            }
        }
        __syncthreads();
        if (wid == 0) {
            for (uint32_t c0 = 0; c0 < nch; c0 += 64) {
                const uint32_t cnt = min(64u, nch - c0);
                const bool in = lane < cnt;
                const uint32_t inc = in ? L.inc[c0 + lane] : kZeros, cef = in ? L.ef[c0 + lane] : 0u;
                uint32_t pos = 0;
                while (pos < cnt && s == s) {  // every pass ends the batch or consumes a chunk
                    const uint32_t bits = __float_as_uint(s), ef = bits >> 23;
                    const bool normal = ef - 1u < 254u;
                    const uint32_t N = normal ? (bits & 0x7fffffu) | 0x800000u : 0u;
                    const bool mine = in && lane >= pos;
                    const bool ok = inc == kZeros || (normal && inc != kMarked && cef == ef);
                    const uint32_t d = mine && ok && inc != kZeros ? inc : 0u;
                    const uint32_t incl = wm::wave_scan_u32(d);
                    const uint64_t off = __ballot(mine && (!ok || N + incl > (1u << 24) - 2u));
                    const uint32_t first = off ? (uint32_t)__builtin_ctzll(off) : cnt;
                    // the exact sum before each chunk up to the offender
                    if (mine && lane <= first)
                        L.pre[c0 + lane] = normal ? ldexpf((float)(N + incl - d), (int)ef - 150) : s;
                    if (normal && first > pos)
                        s = ldexpf((float)(N + (uint32_t)__builtin_amdgcn_readlane((int)incl, (int)first - 1)), (int)ef - 150);
                    if (first == cnt) break;
                    float v[8];
                    f.get8(b0 + (c0 + first) * wm::kSeqBatch + 8 * lane, n, v);
                    s = wm::seq_sum_step(s, v, b0 + c0 + first == 0);
                    pos = first + 1;
                }
            }
            uint32_t h = n;
            if (REACH && s >= r) {
                // the chunk: the last whose sum before it is below r (sums never decrease)
                uint32_t c = 0;
                for (uint32_t c0 = 0; c0 < nch; c0 += 64) {
                    const uint64_t below = __ballot(c0 + lane < nch && L.pre[min(c0 + lane, nch - 1)] < r);
                    if (below) c = c0 + 63 - (uint32_t)__builtin_clzll(below);
                }
                float v[8];
                f.get8(b0 + c * wm::kSeqBatch + 8 * lane, n, v);
                float t = L.pre[c];
                for (uint32_t l = 0; l < 64 && h == n; l++)
#pragma unroll
                    for (uint32_t j = 0; j < 8; j++) {
                        t = t + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v[j]), (int)l));
                        if (h == n && t >= r) h = min(b0 + c * (uint32_t)wm::kSeqBatch + 8 * l + j, n - 1);
                    }
            }
            if (lane == 0) {
                L.s = s;
                L.hit = h;
            }
        }
        __syncthreads();
        s = L.s;
        if (REACH && L.hit != n) {
            *hit = L.hit;
            return s;
        }
    }
    if (REACH) *hit = n;
    return s;
}

__device__ __forceinline__ void write_result(const sample_args &a, uint32_t status, uint32_t id, float total) {
    a.out->id = id;
    a.out->total = total;
    a.out->status = status;
}

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(kSampleThreads) void k_sample_clear(uint32_t *p, uint32_t n) {
    for (uint32_t i = threadIdx.x; i < n; i += kSampleThreads) p[i] = 0;
}

__global__ __launch_bounds__(kSampleThreads) void k_sample_greedy(sample_args a) {
    __shared__ float rv[16];
    __shared__ uint32_t ri[16];
    const uint32_t id = block_argmax_first(plain_terms{a.logits}, a.n, rv, ri);
    if (threadIdx.x == 0) write_result(a, SAMPLE_DONE, id, 0.0f);
}

// Repetition penalty (each history id once: a bit per value of the strip),
// temperature, each workgroup's maximum and, for top-k, the histogram.
// Bound by launch latency and one pass over the logits: 128256 values with
// 600 history ids take 7.5-8.5 us in a kernel trace (one workgroup took
// 100-120 us, the distinct test over the history its largest part).
__global__ __launch_bounds__(kScanThreads) void k_sample_scan(sample_args a) {
    __shared__ uint32_t h[kBins];
    __shared__ uint32_t bits[kStrip / 32];
    __shared__ float red[kScanThreads / 64];
    const uint32_t tid = threadIdx.x;
    const bool hist = a.list;
    const uint64_t lo = (uint64_t)blockIdx.x * a.per, hi = min((uint64_t)a.n, lo + a.per);
    if (hist)
        for (uint32_t i = tid; i < kBins; i += kScanThreads) h[i] = 0;
    // the ids passed as arguments join the device's history for later draws
    if (a.use_rep && blockIdx.x == 0 && tid < a.n_new) a.ids[a.n_ids + tid] = a.new_ids[tid];
    float m = -INFINITY;
    bool nan = false;
    for (uint64_t base = lo; base < hi; base += kStrip) {
        if (a.use_rep) {
            if (tid < kStrip / 32) bits[tid] = 0;
            __syncthreads();
            for (uint32_t j = tid; j < a.n_ids + a.n_new; j += kScanThreads) {
                const uint64_t id = j < a.n_ids ? a.ids[j] : a.new_ids[j - a.n_ids];
                if (id >= base && id < base + kStrip) atomicOr(&bits[(id - base) >> 5], 1u << ((id - base) & 31));
            }
        }
        __syncthreads();
        float v[kStrip / kScanThreads];
#pragma unroll
        for (uint32_t j = 0; j < kStrip / kScanThreads; j++) {
            const uint64_t i = base + tid + j * kScanThreads;
            v[j] = i < hi ? a.logits[i] : -INFINITY;
        }
#pragma unroll
        for (uint32_t j = 0; j < kStrip / kScanThreads; j++) {
            const uint32_t o = tid + j * kScanThreads;
            if (base + o >= hi) continue;
            if (a.use_rep && (bits[o >> 5] >> (o & 31) & 1u)) v[j] = v[j] > 0.0f ? v[j] / a.rep : v[j] * a.rep;
            if (a.use_temp) v[j] = v[j] * a.inv_t;
            a.work[base + o] = v[j];
            nan = nan || isnan(v[j]);
            m = wm_max_nonan(m, v[j]);
            if (hist) atomicAdd(&h[order_key(v[j]) >> 20], 1u);
        }
        __syncthreads();  // the strip's bits are read
    }
    // a NaN among the values top-k sorts leaves the k-th largest unspecified
    if (a.topk_mode == TOPK_THRESHOLD && nan) atomicOr(&a.st->nan, 1u);
    m = wm_block_max_nonan(m, red);  // (its barriers order the histogram too)
    if (tid == 0) a.pmax[blockIdx.x] = m;
    if (hist)
        for (uint32_t i = tid; i < kBins; i += kScanThreads)
            if (h[i]) atomicAdd(&a.hist[i], h[i]);
}

// Top-k: the k-th largest's bin, and this workgroup's values in it and above
// in index order (bin of +0: -0 has the bin below and compares equal).
__global__ __launch_bounds__(kScanThreads) void k_sample_pick(sample_args a) {
    constexpr uint32_t kPer = kBins / kScanThreads;
    __shared__ uint32_t wsum[kScanThreads / 64], bin_s, above_s;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    // thread t takes the t-th group of bins from the top
    const uint32_t g = kScanThreads - 1 - tid;
    uint32_t c[kPer], sum = 0;
#pragma unroll
    for (uint32_t j = 0; j < kPer; j++) {
        c[j] = a.hist[g * kPer + j];
        sum += c[j];
    }
    const uint32_t incl = wm::wave_scan_u32(sum);
    if (lane == 63) wsum[wid] = incl;
    __syncthreads();
    uint32_t above = incl - sum;
    for (uint32_t w = 0; w < wid; w++) above += wsum[w];
    if (above < a.k && above + sum >= a.k) {  // one thread: k <= n
        uint32_t bin = g * kPer, ab = above;
#pragma unroll
        for (int j = (int)kPer - 1; j >= 0; j--) {
            if (ab < a.k && ab + c[j] >= a.k) {
                bin = g * kPer + (uint32_t)j;
                above_s = ab;
            }
            ab += c[j];
        }
        bin_s = bin;
    }
    __syncthreads();
    const uint32_t bin = bin_s;
    if (blockIdx.x == 0 && tid == 0) {
        a.st->bin = bin;
        a.st->above = above_s;
    }
    const uint32_t from = bin == (kKeyPosZero >> 20) ? bin - 1 : bin;
    const uint64_t lo = (uint64_t)blockIdx.x * a.per, hi = min((uint64_t)a.n, lo + a.per);
    uint32_t total = 0;
    for (uint64_t base = lo; base < hi; base += kStrip) {
        const uint64_t i0 = base + 4 * tid;
        uint32_t key[4], keep = 0;
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) {
            key[j] = i0 + j < hi ? order_key(a.work[i0 + j]) : 0u;
            if (i0 + j < hi && (key[j] >> 20) >= from) keep |= 1u << j;
        }
        const uint32_t mine = (uint32_t)__popc(keep), pre = wm::wave_scan_u32(mine);
        __syncthreads();  // the previous strip's counts are read
        if (lane == 63) wsum[wid] = pre;
        __syncthreads();
        uint32_t at = total + pre - mine;
        for (uint32_t w = 0; w < wid; w++) at += wsum[w];
#pragma unroll
        for (uint32_t j = 0; j < 4; j++)
            if (keep >> j & 1u) {
                a.keys[lo + at] = key[j];
                a.vals[lo + at] = (uint32_t)(i0 + j);
                at++;
            }
        for (uint32_t w = 0; w < kScanThreads / 64; w++) total += wsum[w];
    }
    if (tid == 0) a.count[blockIdx.x] = total;
}

// exclusive prefix sum over the workgroup (1024 threads); *total the sum
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t x, uint32_t *wsum, uint32_t *total) {
    const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const uint32_t incl = wm::wave_scan_u32(x);
    wm_sync_lds();
    if (lane == 63) wsum[wid] = incl;
    wm_sync_lds();
    uint32_t before = 0, t = 0;
#pragma unroll
    for (uint32_t w = 0; w < kSampleThreads / 64; w++) {
        before += w < wid ? wsum[w] : 0u;
        t += wsum[w];
    }
    *total = t;
    return before + incl - x;
}

// Top-k's threshold, softmax, top-p and the draw on the listed values, in
// index order in LDS.  Latency-bound (one workgroup, ~20 barriers and the
// serial sums of the kept values): top-k 40 takes 14 us, top-k 1000 37 us.  A
// whole draw of 128256 values with penalty, top-k 40 and top-p: 1209 -> 38
// us, with top-k 1000 1068 -> 61 (the sort of all values, its launches and
// the one-wave sums over 128256 terms gone).
__global__ __launch_bounds__(kSampleThreads) void k_sample_topk(sample_args a) {
    __shared__ uint64_t sorted[4096];  // the list (keys, then indices), later top-p's order
    __shared__ uint32_t kept_i[kListCap];
    __shared__ float kept_p[kListCap];
    __shared__ uint32_t wsum[16], sel_s, bcast_u;
    __shared__ float red[16], bcast;
    static_assert(sizeof(sorted) + 8 * kListCap <= 65536 - 1024, "static LDS");
    static_assert(kMaxParts <= kListCap && kMaxParts <= kSampleThreads, "a part's offset per thread");
    uint32_t *lkey = reinterpret_cast<uint32_t *>(sorted), *lidx = lkey + 4096;
    uint32_t *off = kept_i, *bins = reinterpret_cast<uint32_t *>(kept_p);  // before the filter
    const uint32_t tid = threadIdx.x, wid = tid >> 6, lane = tid & 63;
    const uint32_t bin = a.st->bin, above = a.st->above, nan = a.st->nan;
    const uint32_t mine = tid < a.parts ? a.count[tid] : 0u;
    uint32_t C;
    const uint32_t at = block_excl_scan(mine, wsum, &C);
    off[tid] = at;
    for (uint32_t i = tid; i < kBins; i += kSampleThreads) a.hist[i] = 0;  // for the next draw
    __syncthreads();
    if (tid == 0) a.st->nan = 0;
    if (nan || C > kListCap) {
        if (tid == 0) write_result(a, nan ? SAMPLE_NAN_ORDER : SAMPLE_LIST_FULL, 0, 0.0f);
        return;
    }
    for (uint32_t e = tid; e < C; e += kSampleThreads) {
        uint32_t p = 0;  // the last part whose offset is at most e
        for (uint32_t w = kMaxParts / 2; w; w >>= 1)
            if (p + w < a.parts && off[p + w] <= e) p += w;
        const uint64_t src = (uint64_t)p * a.per + (e - off[p]);
        lkey[e] = a.keys[src];
        lidx[e] = a.vals[src];
    }
    // the k-th largest: among the bin's values the (k - above)-th, by two
    // passes of 10 bits
    uint32_t want = a.k - above, prefix = bin;
    for (int shift = 10; shift >= 0; shift -= 10) {
        __syncthreads();
        bins[tid] = 0;
        __syncthreads();
        for (uint32_t e = tid; e < C; e += kSampleThreads)
            if (lkey[e] >> (shift + 10) == prefix) atomicAdd(&bins[lkey[e] >> shift & 1023u], 1u);
        __syncthreads();
        const uint32_t b = 1023 - tid, cb = bins[b];
        uint32_t tot;
        const uint32_t ab = block_excl_scan(cb, wsum, &tot);
        if (ab < want && ab + cb >= want) {
            sel_s = b;
            bcast_u = ab;
        }
        __syncthreads();
        prefix = prefix << 10 | sel_s;
        want -= bcast_u;
    }
    // kept: not below the k-th largest (+0 and -0 compare equal)
    const uint32_t thr = prefix == kKeyPosZero ? kKeyNegZero : prefix;
    uint32_t K = 0;
    float m = -INFINITY;
    for (uint32_t e0 = 0; e0 < C; e0 += kSampleThreads) {
        const uint32_t e = e0 + tid;
        const bool keep = e < C && lkey[e] >= thr;
        const uint32_t key = keep ? lkey[e] : 0u, idx = keep ? lidx[e] : 0u;
        uint32_t tot;
        const uint32_t p = K + block_excl_scan(keep ? 1u : 0u, wsum, &tot);  // (bins, off read before its barriers)
        if (keep) {
            kept_i[p] = idx;
            kept_p[p] = key_value(key);
            m = wm_max_nonan(m, key_value(key));
        }
        K += tot;
    }
    m = wm_block_max_nonan(m, red);
    if (!isfinite(m)) {
        // every probability is 0: top-p's argmax is index 0, with weight 1
        if (tid == 0) write_result(a, a.topp_mode == TOPP_ONE_HOT ? SAMPLE_DONE : SAMPLE_NOT_POSITIVE, 0,
                                   a.topp_mode == TOPP_ONE_HOT ? 1.0f : 0.0f);
        return;
    }
    __syncthreads();
    for (uint32_t e = tid; e < K; e += kSampleThreads) kept_p[e] = wm_expf(kept_p[e] - m);
    // p *= 1 / Σp (softmax's, then top-p's): exact left-to-right sum
    const auto normalise = [&]() {
        __syncthreads();
        if (wid == 0) {
            const float s = list_sum(kept_p, K);
            if (lane == 0) bcast = s;
        }
        __syncthreads();
        const float sum = bcast;
        if (sum > 0.0f) {
            const float inv = 1.0f / sum;
            for (uint32_t e = tid; e < K; e += kSampleThreads) kept_p[e] *= inv;
        }
    };
    normalise();
    if (a.topp_mode == TOPP_ONE_HOT) {
        __syncthreads();
        const uint32_t am = block_argmax_first(plain_terms{kept_p}, K, red, wsum);
        // u * 1 is reached at the one-hot entry, or at index 0 when it is 0
        if (tid == 0) write_result(a, SAMPLE_DONE, a.unit * 1.0f <= 0.0f ? 0u : kept_i[am], 1.0f);
        return;
    }
    if (a.topp_mode == TOPP_CUT) {
        // descending by probability, equal ones in index order: bitonic sort
        // of (probability bits, ~position)
        uint32_t P = 64;
        while (P < K) P <<= 1;
        __syncthreads();
        for (uint32_t e = tid; e < P; e += kSampleThreads)
            sorted[e] = e < K ? (uint64_t)__float_as_uint(kept_p[e]) << 32 | (uint32_t)~e : 0ull;
        for (uint32_t size = 2; size <= P; size <<= 1)
            for (uint32_t d = size >> 1; d; d >>= 1) {
                __syncthreads();
                for (uint32_t t = tid; t < P / 2; t += kSampleThreads) {
                    const uint32_t i = (t & ~(d - 1)) << 1 | (t & (d - 1)), j = i + d;  // d: a power of two
                    const uint64_t x = sorted[i], y = sorted[j];
                    if ((x < y) == ((i & size) == 0)) {
                        sorted[i] = y;
                        sorted[j] = x;
                    }
                }
            }
        __syncthreads();
        if (wid == 0) {
            float s = 0.0f;
            uint32_t cut = K;
            for (uint32_t b = 0; b < K && cut == K; b += 64) {
                const float x = b + lane < K ? __uint_as_float((uint32_t)(sorted[b + lane] >> 32)) : 0.0f;
                const uint32_t mm = min(64u, K - b);
                for (uint32_t l = 0; l < mm && cut == K; l += 8)
#pragma unroll
                    for (uint32_t j = 0; j < 8; j++) {
                        s = s + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), (int)(l + j)));
                        if (cut == K && b + l + j < K && s >= a.top_p) cut = b + l + j;
                    }
            }
            if (lane == 0) bcast_u = cut == K ? K : cut + 1;  // the entry that reaches p is kept
        }
        __syncthreads();
        const uint64_t last = sorted[bcast_u - 1];
        for (uint32_t e = tid; e < K; e += kSampleThreads)
            if (((uint64_t)__float_as_uint(kept_p[e]) << 32 | (uint32_t)~e) < last) kept_p[e] = 0.0f;
    }
    if (a.topp_mode == TOPP_CUT || a.topp_mode == TOPP_KEEP_ALL) normalise();
    __syncthreads();
    if (wid == 0) {
        const float total = list_sum(kept_p, K);
        if (total <= 0.0f || !isfinite(total)) {
            if (lane == 0) write_result(a, SAMPLE_NOT_POSITIVE, 0, total);
        } else {
            // (the values not kept are zeros: they reach r only if it is 0, at index 0)
            const float r = a.unit * total;
            const uint32_t j = list_first_reach(kept_p, K, r);
            if (lane == 0) write_result(a, SAMPLE_DONE, r <= 0.0f ? 0u : j == K ? a.n - 1 : kept_i[j], total);
        }
    }
}

// The top-k mask and exp(v - max) of all n values (zeros when the maximum is
// not finite).
__global__ __launch_bounds__(kScanThreads) void k_sample_exp(sample_args a) {
    __shared__ float red[kScanThreads / 64];
    const uint32_t tid = threadIdx.x;
    float m = -INFINITY;
    for (uint32_t i = tid; i < a.parts; i += kScanThreads) m = wm_max_nonan(m, a.pmax[i]);
    m = wm_block_max_nonan(m, red);  // the mask keeps the largest, or nothing
    const bool ok = a.topk_mode != TOPK_ALL && isfinite(m);
    const bool mask = a.topk_mode == TOPK_THRESHOLD;
    const float thr = mask ? key_value(a.skeys[a.k - 1]) : 0.0f;
    const uint64_t lo = (uint64_t)blockIdx.x * a.per, hi = min((uint64_t)a.n, lo + a.per);
    for (uint64_t i = lo + tid; i < hi; i += kScanThreads) {
        const float v = a.work[i];
        a.probs[i] = !ok ? 0.0f : wm_expf((mask && v < thr ? -INFINITY : v) - m);
    }
}

// keys of the top-k sort
__global__ __launch_bounds__(kScanThreads) void k_sample_keys_topk(sample_args a) {
    const uint64_t lo = (uint64_t)blockIdx.x * a.per, hi = min((uint64_t)a.n, lo + a.per);
    for (uint64_t i = lo + threadIdx.x; i < hi; i += kScanThreads) a.keys[i] = order_key(a.work[i]);
}

// keys of the top-p sort
__global__ __launch_bounds__(kScanThreads) void k_sample_keys_topp(sample_args a) {
    const float inv = a.st->inv;
    const uint64_t lo = (uint64_t)blockIdx.x * a.per, hi = min((uint64_t)a.n, lo + a.per);
    bool nan = false;
    for (uint64_t i = lo + threadIdx.x; i < hi; i += kScanThreads) {
        const float p = a.probs[i] * inv;
        nan = nan || isnan(p);
        a.keys[i] = order_key(p);
        a.vals[i] = (uint32_t)i;
    }
    if (nan) atomicOr(&a.st->nan, 1u);
}

__device__ __forceinline__ float norm_factor(float sum) { return sum > 0.0f ? 1.0f / sum : 1.0f; }

__device__ void sample_draw(const sample_args &a, const prob_terms &p, block_seq_lds &L) {
    const float total = block_seq<false>(p, a.n, 0.0f, nullptr, L);
    if (total <= 0.0f || !isfinite(total)) {
        if (threadIdx.x == 0) write_result(a, SAMPLE_NOT_POSITIVE, 0, total);
        return;
    }
    const float r = a.unit * total;
    uint32_t j;
    block_seq<true>(p, a.n, r, &j, L);
    if (threadIdx.x == 0) write_result(a, SAMPLE_DONE, r <= 0.0f ? 0u : j == a.n ? a.n - 1 : j, total);
}

// softmax's sum; without a top-p cut also the draw
__global__ __launch_bounds__(kSampleThreads) void k_sample_norm(sample_args a) {
    __shared__ block_seq_lds L;
    __shared__ float rv[16];
    __shared__ uint32_t ri[16];
    // NaN under a top-k that did not go by list (k_sample_topk sees the
    // others'): with top-p the error is k_sample_cut's to give
    const uint32_t nan = a.topk_mode == TOPK_THRESHOLD ? a.st->nan : 0u;
    __syncthreads();
    if (nan && a.topp_mode != TOPP_CUT) {
        if (threadIdx.x == 0) {
            a.st->nan = 0;
            write_result(a, SAMPLE_NAN_ORDER, 0, 0.0f);
        }
        return;
    }
    prob_terms p{a.probs, 1.0f, 1.0f, false, 0.0f, 0u};
    p.inv = norm_factor(block_seq<false>(plain_terms{a.probs}, a.n, 0.0f, nullptr, L));
    if (a.topp_mode == TOPP_CUT) {
        if (threadIdx.x == 0) a.st->inv = p.inv;
        return;
    }
    if (a.topp_mode == TOPP_ONE_HOT) {
        const uint32_t am = block_argmax_first(p, a.n, rv, ri);
        if (threadIdx.x == 0) write_result(a, SAMPLE_DONE, a.unit * 1.0f <= 0.0f ? 0u : am, 1.0f);
        return;
    }
    if (a.topp_mode == TOPP_KEEP_ALL) p.inv2 = norm_factor(block_seq<false>(p, a.n, 0.0f, nullptr, L));
    sample_draw(a, p, L);
}

// top-p's cut in the sorted order, its renormalisation, the draw
__global__ __launch_bounds__(kSampleThreads) void k_sample_cut(sample_args a) {
    __shared__ block_seq_lds L;
    const uint32_t nan = a.st->nan;
    __syncthreads();
    if (nan) {
        if (threadIdx.x == 0) {
            a.st->nan = 0;
            write_result(a, SAMPLE_NAN_ORDER, 0, 0.0f);
        }
        return;
    }
    prob_terms p{a.probs, a.st->inv, 1.0f, true, 0.0f, 0u};
    uint32_t j;
    block_seq<true>(key_terms{a.skeys}, a.n, a.top_p, &j, L);
    const uint32_t last = min(j, a.n - 1);  // the entry that reaches p is kept; all when none does
    p.cut_p = key_value(a.skeys[last]);
    p.cut_i = a.svals[last];
    p.inv2 = norm_factor(block_seq<false>(p, a.n, 0.0f, nullptr, L));
    sample_draw(a, p, L);
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// Rust's `{}` of an f32 for the values the multinomial error can show.
void rust_f32(float v, char *buf, size_t len) {
    if (std::isnan(v)) snprintf(buf, len, "NaN");
    else if (std::isinf(v)) snprintf(buf, len, v > 0 ? "inf" : "-inf");
    else if (v == 0.0f) snprintf(buf, len, std::signbit(v) ? "-0" : "0");
    else snprintf(buf, len, "%.9g", (double)v);
}

}  // namespace

struct wm_sampler {
    wm_ctx *ctx = nullptr;
    int device = 0;
    wm_sampling_params p{};
    uint64_t state = 0;
    std::vector<uint32_t> hist;
    // device workspace for n values (grown on demand)
    void *ws = nullptr;
    size_t ws_bytes = 0;
    uint32_t *d_hist = nullptr;
    size_t d_hist_cap = 0, d_hist_synced = 0;
    // the histogram and the state between kernels (cleared after use), the
    // per-part counts and maxima; and the result in pinned host memory
    uint32_t *d_fixed = nullptr;
    bool fixed_clean = false;
    sample_result *h_out = nullptr;
};

namespace {

uint64_t xorshift_next(uint64_t &s) {  // XorShift64::next_u64 (sampler.rs:26-33)
    uint64_t x = s;
    x ^= x << 13;
    x ^= x >> 7;
    x ^= x << 17;
    s = x;
    return x;
}

bool is_greedy(const wm_sampling_params &p) {  // SamplingParams::is_greedy (sampler.rs:71-78)
    return std::fabs(p.temperature) < 1e-9f && !p.has_top_k && !p.has_top_p &&
           !p.has_repetition_penalty;
}

size_t sort_temp_bytes(uint32_t n, hipStream_t s) {
    size_t a = 0, b = 0;
    rocprim::radix_sort_keys_desc(nullptr, a, (uint32_t *)nullptr, (uint32_t *)nullptr, n, 0, 32, s);
    rocprim::radix_sort_pairs_desc(nullptr, b, (uint32_t *)nullptr, (uint32_t *)nullptr,
                                   (uint32_t *)nullptr, (uint32_t *)nullptr, n, 0, 32, s);
    return a > b ? a : b;
}

}  // namespace

// Sample from n logits at d_logits (device).  Called with the sampler's
// context current.
wm_status wm_sampler_run(wm_sampler *sp, const float *d_logits, uint32_t n, uint32_t *out_id) {
    wm_ctx *ctx = sp->ctx;
    hipStream_t s = ctx->stream;
    const wm_sampling_params &p = sp->p;
    const bool greedy = is_greedy(p);
    if (n == 0) {
        if (greedy) return wm_set_error(ctx, WM_E_PARSE, "sample: empty logits");
        return wm_set_error(ctx, WM_E_PARSE,
                            "multinomial: probabilities do not sum to a positive finite value (0)");
    }
    // parts of a multiple of kStrip values, at most kMaxParts of them
    const uint64_t strips = ((uint64_t)n + kStrip - 1) / kStrip;
    const uint32_t per = (uint32_t)((strips + kMaxParts - 1) / kMaxParts * kStrip);
    const uint32_t parts = (uint32_t)(((uint64_t)n + per - 1) / per);
    const size_t tmp_bytes = sort_temp_bytes(n, s);
    const size_t f = align256((size_t)n * 4);
    const size_t need = 6 * f + align256(tmp_bytes);
    WM_HIP(ctx, hipSetDevice(sp->device));
    if (need > sp->ws_bytes) {
        WM_HIP(ctx, hipStreamSynchronize(s));
        if (sp->ws) WM_HIP(ctx, hipFree(sp->ws));
        sp->ws = nullptr;
        sp->ws_bytes = 0;
        WM_HIP(ctx, hipMalloc(&sp->ws, need));
        sp->ws_bytes = need;
    }
    constexpr size_t kStateWords = 64;
    static_assert(sizeof(sample_state) <= kStateWords * 4, "state slot");
    if (!sp->d_fixed) {
        WM_HIP(ctx, hipMalloc((void **)&sp->d_fixed, (kBins + kStateWords + 2 * kMaxParts) * 4));
        sp->fixed_clean = false;
    }
    if (!sp->h_out) WM_HIP(ctx, hipHostMalloc((void **)&sp->h_out, sizeof(sample_result), hipHostMallocMapped));
    if (!sp->fixed_clean) {
        hipLaunchKernelGGL(k_sample_clear, dim3(1), dim3(kSampleThreads), 0, s, sp->d_fixed,
                           (uint32_t)(kBins + kStateWords));
        WM_HIP(ctx, hipGetLastError());
    }
    sp->fixed_clean = false;  // until this draw has ended
    uint8_t *b = (uint8_t *)sp->ws;
    sample_args a{};
    a.logits = d_logits;
    a.n = n;
    a.parts = parts;
    a.per = per;
    a.work = (float *)b;
    a.probs = (float *)(b + f);
    a.keys = (uint32_t *)(b + 2 * f);
    a.vals = (uint32_t *)(b + 3 * f);
    uint32_t *skeys = (uint32_t *)(b + 4 * f), *svals = (uint32_t *)(b + 5 * f);
    a.skeys = skeys;
    a.svals = svals;
    a.hist = sp->d_fixed;
    a.st = (sample_state *)(sp->d_fixed + kBins);
    a.count = sp->d_fixed + kBins + kStateWords;
    a.pmax = (float *)(a.count + kMaxParts);
    WM_HIP(ctx, hipHostGetDevicePointer((void **)&a.out, sp->h_out, 0));
    void *tmp = b + 6 * f;
    // repetition penalty (sampler.rs:151-164): history on the device, the
    // newest ids as arguments (k_sample_scan appends them)
    const float r = p.repetition_penalty;
    a.use_rep = !greedy && p.has_repetition_penalty && !(r <= 0.0f || std::fabs(r - 1.0f) < 1e-9f) &&
                !sp->hist.empty();
    a.rep = r;
    if (a.use_rep) {
        const size_t len = sp->hist.size();
        if (len > 0xffffffffull - kNewIds) return wm_set_error(ctx, WM_E_SHAPE, "sample: %zu history ids", len);
        if (len > sp->d_hist_cap) {
            WM_HIP(ctx, hipStreamSynchronize(s));
            if (sp->d_hist) WM_HIP(ctx, hipFree(sp->d_hist));
            sp->d_hist = nullptr;
            sp->d_hist_cap = sp->d_hist_synced = 0;
            const size_t cap = len * 2 + 256;
            WM_HIP(ctx, hipMalloc((void **)&sp->d_hist, cap * 4));
            sp->d_hist_cap = cap;
        }
        if (len - sp->d_hist_synced > kNewIds) {
            // the copy reads host memory now (pageable): the vector may grow later
            WM_HIP(ctx, hipMemcpy(sp->d_hist + sp->d_hist_synced, sp->hist.data() + sp->d_hist_synced,
                                  (len - sp->d_hist_synced) * 4, hipMemcpyHostToDevice));
            sp->d_hist_synced = len;
        }
        a.n_ids = (uint32_t)sp->d_hist_synced;
        a.n_new = (uint32_t)(len - sp->d_hist_synced);
        for (uint32_t i = 0; i < a.n_new; i++) a.new_ids[i] = sp->hist[a.n_ids + i];
    }
    a.ids = sp->d_hist;
    // temperature (sampler.rs:166-176)
    const float t = p.temperature;
    a.use_temp = !greedy && !(t <= 0.0f || std::fabs(t - 1.0f) < 1e-9f);
    a.inv_t = 1.0f / t;
    // top-k (sampler.rs:201-223), k clamped to n
    a.topk_mode = TOPK_NONE;
    if (!greedy && p.has_top_k) {
        const uint64_t k = p.top_k < n ? p.top_k : n;
        a.topk_mode = k == 0 ? TOPK_ALL : (k == n ? TOPK_NONE : TOPK_THRESHOLD);
        a.k = (uint32_t)k;
        // At least k values are listed, so a longer list than it holds would be
        // made in vain (128256 values, a draw: top-k 20000 205 -> 183 us, top-k
        // 4500 with top-p 331 -> 309).
        a.list = a.topk_mode == TOPK_THRESHOLD && a.k <= kListCap;
    }
    // top-p (sampler.rs:254-311)
    a.topp_mode = TOPP_NONE;
    a.top_p = p.top_p;
    if (!greedy && p.has_top_p) {
        const float tp = p.top_p;
        if (tp <= 0.0f) a.topp_mode = TOPP_ONE_HOT;
        else if (tp >= 1.0f) a.topp_mode = TOPP_NONE;
        else if (std::isnan(tp)) a.topp_mode = TOPP_KEEP_ALL;  // never reached: every entry kept
        else a.topp_mode = TOPP_CUT;
    }
    // the draw the multinomial would consume (the state advances only if it runs)
    uint64_t next_state = sp->state;
    a.unit = (float)(xorshift_next(next_state) >> 40) / (float)(1ull << 24);

    const dim3 wide(parts), narrow(1);
    sp->h_out->status = SAMPLE_RUNNING;
    bool listed = false;
    if (greedy) {
        hipLaunchKernelGGL(k_sample_greedy, narrow, dim3(kSampleThreads), 0, s, a);
    } else {
        hipLaunchKernelGGL(k_sample_scan, wide, dim3(kScanThreads), 0, s, a);
        if (a.list) {
            hipLaunchKernelGGL(k_sample_pick, wide, dim3(kScanThreads), 0, s, a);
            hipLaunchKernelGGL(k_sample_topk, narrow, dim3(kSampleThreads), 0, s, a);
            WM_HIP(ctx, hipGetLastError());
            WM_HIP(ctx, hipStreamSynchronize(s));
            listed = sp->h_out->status != SAMPLE_LIST_FULL;
        }
        if (!listed) {
            size_t tb = tmp_bytes;
            sp->h_out->status = SAMPLE_RUNNING;
            if (a.topk_mode == TOPK_THRESHOLD) {
                hipLaunchKernelGGL(k_sample_keys_topk, wide, dim3(kScanThreads), 0, s, a);
                WM_HIP(ctx, rocprim::radix_sort_keys_desc(tmp, tb, a.keys, skeys, n, 0, 32, s));
            }
            hipLaunchKernelGGL(k_sample_exp, wide, dim3(kScanThreads), 0, s, a);
            hipLaunchKernelGGL(k_sample_norm, narrow, dim3(kSampleThreads), 0, s, a);
            if (a.topp_mode == TOPP_CUT) {
                hipLaunchKernelGGL(k_sample_keys_topp, wide, dim3(kScanThreads), 0, s, a);
                WM_HIP(ctx, rocprim::radix_sort_pairs_desc(tmp, tb, a.keys, skeys, a.vals, svals, n, 0, 32, s));
                hipLaunchKernelGGL(k_sample_cut, narrow, dim3(kSampleThreads), 0, s, a);
            }
        }
    }
    if (!listed) {
        WM_HIP(ctx, hipGetLastError());
        WM_HIP(ctx, hipStreamSynchronize(s));
    }
    const sample_result st = *sp->h_out;
    sp->fixed_clean = st.status != SAMPLE_RUNNING;
    if (a.use_rep && sp->fixed_clean) sp->d_hist_synced = sp->hist.size();
    if (st.status == SAMPLE_NOT_POSITIVE) {
        char v[32];
        rust_f32(st.total, v, sizeof v);
        return wm_set_error(ctx, WM_E_PARSE,
                            "multinomial: probabilities do not sum to a positive finite value (%s)", v);
    }
    if (st.status == SAMPLE_NAN_ORDER)
        return wm_set_error(ctx, WM_E_NONFINITE,
                            a.topp_mode == TOPP_CUT && a.topk_mode != TOPK_THRESHOLD
                                ? "sample: NaN probabilities under top-p (their order is unspecified)"
                                : "sample: NaN values under top-k or top-p (their order is unspecified)");
    if (st.status != SAMPLE_DONE) return wm_set_error(ctx, WM_E_STATE, "sample: did not finish");
    if (!greedy) sp->state = next_state;
    *out_id = st.id;
    return WM_OK;
}

wm_ctx *wm_sampler_ctx(const wm_sampler *sp) { return sp ? sp->ctx : nullptr; }

extern "C" {

wm_status wm_sampler_create(wm_ctx *ctx, const wm_sampling_params *params, uint64_t seed,
                            wm_sampler **out) {
    if (!ctx || !params || !out) return WM_E_ARG;
    wm_sampler *sp = new wm_sampler();
    sp->ctx = ctx;
    sp->device = ctx->device;
    sp->p = *params;
    sp->state = seed ? seed : 0xdeadbeefcafebabeull;  // XorShift64::new (sampler.rs:18-25)
    *out = sp;
    return WM_OK;
}

void wm_sampler_destroy(wm_sampler *sp) {
    if (!sp) return;
    if (hipSetDevice(sp->device) == hipSuccess) {
        if (sp->ws) (void)hipFree(sp->ws);
        if (sp->d_hist) (void)hipFree(sp->d_hist);
        if (sp->d_fixed) (void)hipFree(sp->d_fixed);
        if (sp->h_out) (void)hipHostFree(sp->h_out);
    }
    delete sp;
}

wm_status wm_sampler_observe(wm_sampler *sp, uint32_t id) {
    if (!sp) return WM_E_ARG;
    sp->hist.push_back(id);
    return WM_OK;
}

wm_status wm_sampler_checkpoint(const wm_sampler *sp, uint64_t *rng_state, uint64_t *history_len) {
    if (!sp || !rng_state || !history_len) return WM_E_ARG;
    *rng_state = sp->state;
    *history_len = sp->hist.size();
    return WM_OK;
}

wm_status wm_sampler_rollback(wm_sampler *sp, uint64_t rng_state, uint64_t history_len) {
    if (!sp) return WM_E_ARG;
    if (history_len > sp->hist.size())
        return wm_set_error(sp->ctx, WM_E_ARG, "sampler rollback: history length %llu beyond %zu",
                            (unsigned long long)history_len, sp->hist.size());
    sp->state = rng_state;
    sp->hist.resize(history_len);
    if (sp->d_hist_synced > history_len) sp->d_hist_synced = history_len;
    return WM_OK;
}

wm_status wm_sampler_sample_dev(wm_sampler *sp, const float *d_logits, size_t n, uint32_t *out_id) {
    if (!sp || !out_id || (n && !d_logits)) return WM_E_ARG;
    if (n > 0xffffffffull) return wm_set_error(sp->ctx, WM_E_SHAPE, "sample: %zu logits", n);
    return wm_sampler_run(sp, d_logits, (uint32_t)n, out_id);
}

wm_status wm_sampler_sample(wm_sampler *sp, const float *logits, size_t n, uint32_t *out_id) {
    if (!sp || !out_id || (n && !logits)) return WM_E_ARG;
    if (n > 0xffffffffull) return wm_set_error(sp->ctx, WM_E_SHAPE, "sample: %zu logits", n);
    wm_ctx *ctx = sp->ctx;
    void *d = nullptr;
    if (n) {
        wm_status st = wm_ctx_scratch(ctx, n * 4, &d);
        if (st) return st;
        WM_HIP(ctx, hipSetDevice(sp->device));
        WM_HIP(ctx, hipMemcpyAsync(d, logits, n * 4, hipMemcpyHostToDevice, ctx->stream));
    }
    return wm_sampler_run(sp, (const float *)d, (uint32_t)n, out_id);
}

}  // extern "C"
