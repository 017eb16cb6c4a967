// Selection shared by the float retrieval paths: the k best of a row of fp32 scores in
// descending order, equal scores in list order.  One workgroup per row; a score travels as an
// order-preserving 32-bit key that can be turned back into the score, so a row is one word per
// candidate.  Included by the translation units that launch it.
#pragma once

#include "common.h"

namespace {

constexpr int kMaxTopk = 4096;  // winners held in LDS: 8 bytes each (32 KiB)
constexpr int kCrowd = 64;      // entries a bin may hold on the direct path
constexpr int kBucketMax = 48;  // entries a bucket may hold when the winners are ordered afterwards
constexpr int kMaxRegKeys = 16; // keys a thread keeps in registers: rows of up to 16384 candidates

// Order-preserving key of a score: larger score <-> larger key.  0 is reserved for "no
// candidate", 1 for NaN (below every number, above nothing else).
__device__ __forceinline__ uint32_t score_key(float s)
{
    if (s != s) return 1u;
    const uint32_t u = __float_as_uint(s);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// The score of a key (a NaN for key 1).
__device__ __forceinline__ float key_score(uint32_t k)
{
    return __uint_as_float((k & 0x80000000u) ? k & 0x7fffffffu : ~k);
}

// A finite number that orders like the key, for dividing the rows' range into equal widths.
__device__ __forceinline__ float key_place(uint32_t k)
{
    const float big = 3.402823466e38f;
    const float v = key_score(k);
    return k == 1u ? -big : (v > big ? big : (v < -big ? -big : v));
}

// Keys of a row lie at a pitch of whole 64-byte lines: every thread loads its keys as 16-byte pieces.
inline int64_t key_pitch(int64_t n) { return (n + 15) & ~(int64_t)15; }

struct SortArgs {
    const uint32_t* keys;   // [B] rows of max_n keys, `pitch` apart; 16-byte aligned
    int64_t pitch;
    const int32_t* idx;     // [B][max_n] what a list position stands for, or null: the position itself
    int max_n, topk, cap;   // cap: entries the search orders in LDS, a power of two
    int32_t* out_idx;       // [B][topk]
    float* out_score;       // [B][topk]
};

// Maximum over the 64 lanes, in every lane: exchanges inside a row of 16 lanes, then the last lane
// of a row broadcast into the next rows (a few cycles each; a shuffle is a trip through the LDS pipe).
__device__ __forceinline__ uint32_t wave_max(uint32_t v)
{
    auto step = [&](uint32_t o) { v = o > v ? o : v; };
    step((uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0xB1, 0xf, 0xf, false));   // quad_perm [1,0,3,2]
    step((uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x4E, 0xf, 0xf, false));   // quad_perm [2,3,0,1]
    step((uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x141, 0xf, 0xf, false));  // row_half_mirror
    step((uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x140, 0xf, 0xf, false));  // row_mirror
    step((uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x142, 0xa, 0xf, false));  // row_bcast:15
    step((uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x143, 0xc, 0xf, false));  // row_bcast:31
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Exclusive prefix sum of one int per thread over a workgroup of NT threads.
template <int NT>
__device__ __forceinline__ int scan_wg(int v, int* wsum, int* total)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int inc = v;
    inc += __builtin_amdgcn_update_dpp(0, inc, 0x111, 0xf, 0xf, false);  // row_shr:1
    inc += __builtin_amdgcn_update_dpp(0, inc, 0x112, 0xf, 0xf, false);  // row_shr:2
    inc += __builtin_amdgcn_update_dpp(0, inc, 0x114, 0xf, 0xf, false);  // row_shr:4
    inc += __builtin_amdgcn_update_dpp(0, inc, 0x118, 0xf, 0xf, false);  // row_shr:8
    inc += __builtin_amdgcn_update_dpp(0, inc, 0x142, 0xa, 0xf, false);  // row_bcast:15
    inc += __builtin_amdgcn_update_dpp(0, inc, 0x143, 0xc, 0xf, false);  // row_bcast:31
    __syncthreads();
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    int base = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) {
        const int x = wsum[i];
        if (i < w) base += x;
        tot += x;
    }
    *total = tot;
    return base + inc - v;
}

// Direct path.  The row's range of scores is divided into 4 NT bins of equal width, the keys are
// counted per bin, a prefix sum over the bins (best first) says where each bin's entries go, and the
// entries of the bins that start before place k are put there and ranked among the few that share
// their bin.  Returns false, with nothing written, when such a bin holds more than kCrowd entries
// (many equal scores, or a range stretched by outliers).
// What bounds it is its chain of barriers and LDS round trips, not bytes: one pass over the keys
// replaces the search for the k-th key digit by digit, the compaction and the ordering (4 + 2 + 3
// passes of counting, scanning and placing).  8000 candidates, k = 3000, two rows: 21.0 us for the
// digit search, 8.1 us like this on one workgroup per row, 6.8 us with the places shared by three.
template <int NT, int PER>
__device__ __forceinline__ bool topk_direct(const SortArgs& a, const uint32_t (&kreg)[PER], uint32_t* bins,
                                            unsigned long long* win, int* wsum, uint32_t (*range)[NT / 64],
                                            int* s_two)
{
    constexpr int kBins = 4 * NT;
    const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    uint32_t hi = 0u, lo = 0u;  // largest key and largest complement of a key
#pragma unroll
    for (int e = 0; e < PER; ++e) {
        hi = kreg[e] > hi ? kreg[e] : hi;
        lo = kreg[e] != 0u && ~kreg[e] > lo ? ~kreg[e] : lo;
    }
    hi = wave_max(hi);
    lo = wave_max(lo);
    if (lane == 0) {
        range[0][w] = hi;
        range[1][w] = lo;
    }
    reinterpret_cast<uint4*>(bins)[tid] = make_uint4(0u, 0u, 0u, 0u);
    if (tid < 2) s_two[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) {
        hi = range[0][i] > hi ? range[0][i] : hi;
        lo = range[1][i] > lo ? range[1][i] : lo;
    }
    const float top = key_place(hi), width = top - key_place(~lo);
    // an infinite width (range over the float limits) puts everything into one bin: the other path's case
    const float scale = width > 0.0f ? (float)(kBins - 1) / width : 0.0f;
    auto bin_of = [&](uint32_t k) {
        const float at = (top - key_place(k)) * scale;  // not a number where the range is infinite: bin 0
        return at > 0.0f ? (int)(at < (float)(kBins - 1) ? at : (float)(kBins - 1)) : 0;
    };
    int bin[PER], at[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) {
        bin[e] = bin_of(kreg[e]);
        at[e] = 0;
        if (kreg[e] != 0u) at[e] = (int)atomicAdd(&bins[bin[e]], 1u);
    }
    __syncthreads();
    const uint4 c = reinterpret_cast<const uint4*>(bins)[tid];
    int n_valid;
    const int before = scan_wg<NT>((int)(c.x + c.y + c.z + c.w), wsum, &n_valid);
    const int kk = n_valid < a.topk ? n_valid : a.topk;
    // (first place << 16 | entries) per bin; both fit: a row on this path has at most 16384 candidates
    const uint32_t cnt[4] = {c.x, c.y, c.z, c.w};
    uint32_t packed[4];
    // this workgroup's share of the places: the entries of the bins that start in [lo_at, hi_at)
    const int share = (kk + (int)gridDim.y - 1) / (int)gridDim.y;
    const int lo_at = (int)blockIdx.y * share;
    const int hi_at = lo_at >= kk ? lo_at : (lo_at + share < kk ? lo_at + share : kk);
    int first = before, end_lo = -1, end_hi = -1;
    bool crowded = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        packed[i] = (uint32_t)first << 16 | cnt[i];
        crowded |= first < kk && cnt[i] > (uint32_t)kCrowd;
        if (first < lo_at) end_lo = first + (int)cnt[i];
        if (first < hi_at) end_hi = first + (int)cnt[i];
        first += (int)cnt[i];
    }
    reinterpret_cast<uint4*>(bins)[tid] = make_uint4(packed[0], packed[1], packed[2], packed[3]);
    // where the last bins that start before lo_at and before hi_at end; one thread has each
    if (before < lo_at && first >= lo_at) s_two[0] = end_lo;
    if (before < hi_at && first >= hi_at) s_two[1] = end_hi;
    if (__syncthreads_or(crowded)) return false;
#pragma unroll
    for (int e = 0; e < PER; ++e) {
        if (kreg[e] == 0u) continue;
        const int f = (int)(bins[bin[e]] >> 16);
        if (f >= lo_at && f < hi_at) win[f - lo_at + at[e]] = ((unsigned long long)kreg[e] << 32) | (uint32_t)(~(uint32_t)(tid * PER + e));
    }
    __syncthreads();
    const int end = s_two[1];
    for (int i = s_two[0] + tid; i < end; i += NT) {
        const unsigned long long x = win[i - lo_at];
        const uint32_t k = (uint32_t)(x >> 32);
        const int pos = (int)(~(uint32_t)x);
        const int32_t id = a.idx ? a.idx[(int64_t)b * a.max_n + pos] : pos;
        const uint32_t p = bins[bin_of(k)];
        const int f = (int)(p >> 16), n = (int)(p & 0xffffu);
        int rank = f;  // entries of the bin that go before this one come first
        for (int j = 0; j < n; ++j) rank += win[f - lo_at + j] > x;
        if (rank < kk) {
            a.out_idx[(int64_t)b * a.topk + rank] = id;
            a.out_score[(int64_t)b * a.topk + rank] = k == 1u ? __uint_as_float(0x7fc00000u) : key_score(k);
        }
    }
    for (int t = kk + (int)blockIdx.y * NT + tid; t < a.topk; t += NT * (int)gridDim.y) {
        a.out_idx[(int64_t)b * a.topk + t] = -1;
        a.out_score[(int64_t)b * a.topk + t] = 0.0f;
    }
    return true;
}

// Any row.  Four 8-bit radix passes find the k-th largest key, winners go to LDS at slots from one
// prefix sum (keys above the threshold, then the ties in list order), and (key, position) pairs are
// ordered: equal-width buckets over [threshold, largest key], or bitonic networks and pairwise merges
// where a bucket is crowded.  PER = 0: keys are re-read from memory in every phase (rows longer than
// the registers hold).
template <int NT, int PER>
__device__ void topk_search(const SortArgs& a, const uint32_t (&kreg)[PER ? PER : 1], uint32_t* lds,
                            unsigned long long* win, int* wsum, int* s_two)
{
    constexpr bool REG = PER > 0;
    constexpr int kBuckets = NT;  // one per thread
    int* hist = reinterpret_cast<int*>(lds);        // 256
    int* bcount = reinterpret_cast<int*>(lds);      // kBuckets each, after the search
    int* bfill = bcount + kBuckets;
    int* bbase = bfill + kBuckets;
    const int b = blockIdx.x;
    const uint32_t* keys = a.keys + b * a.pitch;
    const int tid = threadIdx.x, lane = tid & 63;
    // f(chunk, key) over the thread's keys; uniform control flow.  Without registers chunk e covers
    // list positions e * NT + tid.
    auto for_chunks = [&](auto&& f) {
        if constexpr (REG) {
#pragma unroll
            for (int e = 0; e < PER; ++e) f(e, kreg[e]);
        } else {
            for (int e = 0; e * NT < a.max_n; ++e) {
                const int i = e * NT + tid;
                f(e, i < a.max_n ? keys[i] : 0u);
            }
        }
    };

    // candidates present
    int mine = 0;
    for_chunks([&](int, uint32_t k) { mine += k != 0u; });
    int n_valid;
    (void)scan_wg<NT>(mine, wsum, &n_valid);
    const int kk = n_valid < a.topk ? n_valid : a.topk;

    // ---- radix search, 8 bits a pass, for the kk-th largest key among the candidates ----
    uint32_t prefix = 0, mask = 0;
    int need = kk;
    for (int shift = 24; shift >= 0 && kk > 0; shift -= 8) {
        if (tid < 256) hist[tid] = 0;
        __syncthreads();
        for_chunks([&](int, uint32_t k) {
            const bool in = k != 0u && (k & mask) == prefix;
            const int d = (k >> shift) & 255;
            // scores of one magnitude share their leading digits: when a whole wave holds one
            // digit its first lane adds the count (64 lanes adding to one LDS word serialise)
            const unsigned long long act = __ballot(in);
            if (act != 0ull) {
                const int first = __ffsll((long long)act) - 1;
                const int d0 = __shfl(d, first);
                if (__ballot(in && d == d0) == act) {
                    if (lane == first) atomicAdd(&hist[d0], __popcll(act));
                } else if (in) {
                    atomicAdd(&hist[d], 1);
                }
            }
        });
        __syncthreads();
        // digits in descending order, one per thread: the chosen digit is where the running
        // count first reaches `need`
        const int cnt = tid < 256 ? hist[255 - tid] : 0;
        int all;
        const int before = scan_wg<NT>(cnt, wsum, &all);
        if (tid < 256 && before < need && before + cnt >= need) {
            s_two[0] = 255 - tid;
            s_two[1] = need - before;  // still to take among keys with this digit
        }
        __syncthreads();
        prefix |= (uint32_t)s_two[0] << shift;
        mask |= 255u << shift;
        need = s_two[1];
        __syncthreads();
    }
    const uint32_t thr = prefix;  // the kk-th largest key; `need` of the keys equal to it are taken

    // ---- winners into LDS: every key above the threshold, then the first `need` equal to it.
    //      Slots come from a prefix sum over the list (both counts packed into one scan), not
    //      from a shared counter: thousands of increments of one LDS word would serialise ----
    for (int i = tid; i < a.cap; i += NT) win[i] = 0ull;
    __syncthreads();
    const int n_gt = kk - need;  // keys above the threshold
    int gt_before = 0, eq_before = 0;
    if (kk > 0) {
        if constexpr (REG) {
            int my_gt = 0, my_eq = 0;
#pragma unroll
            for (int e = 0; e < PER; ++e) {
                my_gt += kreg[e] > thr && kreg[e] != 0u;
                my_eq += kreg[e] == thr && kreg[e] != 0u;
            }
            int total;
            const int before = scan_wg<NT>(my_gt | (my_eq << 16), wsum, &total);
            int gt_at = before & 0xffff, eq_at = before >> 16;
#pragma unroll
            for (int e = 0; e < PER; ++e) {
                const uint32_t k = kreg[e];
                const int i = tid * PER + e;
                int slot = -1;
                if (k > thr && k != 0u) slot = gt_at++;
                else if (k == thr && k != 0u) {
                    if (eq_at < need) slot = n_gt + eq_at;
                    ++eq_at;
                }
                if (slot >= 0) win[slot] = ((unsigned long long)k << 32) | (uint32_t)(~(uint32_t)i);
            }
        } else {
            for_chunks([&](int e, uint32_t k) {
                const int i = e * NT + tid;
                const bool gt = k > thr && k != 0u;
                const bool eq = k == thr && k != 0u;
                int total;
                const int before = scan_wg<NT>((gt ? 1 : 0) | (eq ? 1 << 16 : 0), wsum, &total);
                const int eq_rank = eq_before + (before >> 16);
                int slot = -1;
                if (gt) slot = gt_before + (before & 0xffff);
                else if (eq && eq_rank < need) slot = n_gt + eq_rank;
                if (slot >= 0) win[slot] = ((unsigned long long)k << 32) | (uint32_t)(~(uint32_t)i);
                gt_before += total & 0xffff;
                eq_before += total >> 16;
            });
        }
    }
    __syncthreads();

    // ---- order the winners, descending: larger key first, then smaller position ----
    // The winners' keys lie in [thr, kmax]; equal-width buckets over that range (descending), a
    // prefix sum over the bucket counts, every winner dropped into its bucket, then ranked among the
    // few entries that share it.
    constexpr int kPer = REG && NT * PER < kMaxTopk ? PER : kMaxTopk / NT;  // entries per thread at the largest cap
    uint32_t kmax = 0u;
    unsigned long long x[kPer];
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        const int i = tid + e * NT;
        x[e] = i < kk ? win[i] : 0ull;
        const uint32_t k = (uint32_t)(x[e] >> 32);
        kmax = k > kmax ? k : kmax;
    }
    kmax = wave_max(kmax);
    bcount[tid] = 0;
    bfill[tid] = 0;
    if (lane == 0) wsum[tid >> 6] = (int)kmax;
    __syncthreads();
    for (int w = 0; w < NT / 64; ++w) kmax = (uint32_t)wsum[w] > kmax ? (uint32_t)wsum[w] : kmax;
    const uint32_t range = kmax > thr ? kmax - thr : 0u;
    const int bits = range ? 32 - __builtin_clz(range) : 0;
    constexpr int kBucketBits = __builtin_ctz(kBuckets);
    const int bshift = bits > kBucketBits ? bits - kBucketBits : 0;
    int bucket[kPer];
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        const int i = tid + e * NT;
        bucket[e] = -1;
        if (i < kk) {
            bucket[e] = (kBuckets - 1) - (int)(((uint32_t)(x[e] >> 32) - thr) >> bshift);
            atomicAdd(&bcount[bucket[e]], 1);
        }
    }
    __syncthreads();
    const int my_count = bcount[tid];
    int all_winners;
    const int my_base = scan_wg<NT>(my_count, wsum, &all_winners);
    const bool crowded = __syncthreads_or(my_count > kBucketMax);
    if (!crowded) {
        bbase[tid] = my_base;
        __syncthreads();
#pragma unroll
        for (int e = 0; e < kPer; ++e)
            if (bucket[e] >= 0) win[bbase[bucket[e]] + atomicAdd(&bfill[bucket[e]], 1)] = x[e];
        __syncthreads();
        int dst[kPer];
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
            dst[e] = -1;
            if (bucket[e] >= 0) {
                const int first = bbase[bucket[e]], n = bcount[bucket[e]];
                int ahead = 0;  // entries of the bucket that go before this one
                for (int j = 0; j < n; ++j) ahead += win[first + j] > x[e];
                dst[e] = first + ahead;
            }
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < kPer; ++e)
            if (dst[e] >= 0) win[dst[e]] = x[e];
        __syncthreads();
    } else {
        // (a) bitonic networks over aligned segments of 256 entries, every segment descending;
        // (b) sorted runs merged pairwise: an entry's place in the merged run is its place in its
        //     own run plus the number of entries of the sibling run that go before it (binary
        //     search; the left run wins ties, which only the empty slots have).  For 4096 entries
        //     that is 36 + 2 * 4 barriers where one network over everything takes 78.
        const int seg = a.cap < 256 ? a.cap : 256;
        for (int size = 2; size <= seg; size <<= 1) {
            for (int stride = size >> 1; stride > 0; stride >>= 1) {
                for (int t = tid; t < a.cap / 2; t += NT) {
                    const int lo = 2 * t - (t & (stride - 1));
                    const int hi = lo + stride;
                    const bool desc = size == seg || (lo & size) == 0;
                    const unsigned long long p = win[lo], q = win[hi];
                    if ((p < q) == desc) {
                        win[lo] = q;
                        win[hi] = p;
                    }
                }
                __syncthreads();
            }
        }
        for (int run = seg; run < a.cap; run <<= 1) {
            int dst[kPer];
            const int sh = __builtin_ctz(run);
#pragma unroll
            for (int e = 0; e < kPer; ++e) {
                const int i = tid + e * NT;
                dst[e] = -1;
                if (i < a.cap) {
                    x[e] = win[i];
                    const int r = i >> sh, at = i & (run - 1);
                    const unsigned long long* sib = win + (r ^ 1) * run;
                    const bool left = (r & 1) == 0;
                    int lo = 0, hi = run;  // entries of the sibling run that go before x[e]
                    while (lo < hi) {
                        const int mid = (lo + hi) >> 1;
                        const unsigned long long o = sib[mid];
                        if (o > x[e] || (!left && o == x[e])) lo = mid + 1;
                        else hi = mid;
                    }
                    dst[e] = (r >> 1) * 2 * run + at + lo;
                }
            }
            __syncthreads();
#pragma unroll
            for (int e = 0; e < kPer; ++e)
                if (dst[e] >= 0) win[dst[e]] = x[e];
            __syncthreads();
        }
    }

    for (int t = tid; t < a.topk; t += NT) {
        int32_t oi = -1;
        float os = 0.0f;
        if (t < kk) {
            const int pos = (int)(~(uint32_t)(win[t] & 0xffffffffull));
            const uint32_t k = (uint32_t)(win[t] >> 32);
            oi = a.idx ? a.idx[(int64_t)b * a.max_n + pos] : pos;
            os = k == 1u ? __uint_as_float(0x7fc00000u) : key_score(k);
        }
        a.out_idx[(int64_t)b * a.topk + t] = oi;
        a.out_score[(int64_t)b * a.topk + t] = os;
    }
}

// grid = (rows, workgroups per row); dynamic LDS: the winners' array.  Thread t holds list positions t * PER ..
// t * PER + PER - 1 (consecutive, so that one prefix sum over per-thread counts orders the list).
template <int NT, int PER>
__global__ __launch_bounds__(NT) void topk_kernel(SortArgs a)
{
    extern __shared__ unsigned long long win[];  // [cap] (key << 32) | ~position
    __shared__ __align__(16) uint32_t bins[4 * NT];
    __shared__ int wsum[NT / 64];
    __shared__ uint32_t range[2][NT / 64];
    __shared__ int s_two[2];
    if constexpr (PER > 0) {
        static_assert(PER == 1 || PER % 4 == 0, "16-byte loads");
        uint32_t kreg[PER];
        const uint32_t* keys = a.keys + blockIdx.x * a.pitch;
        const int first = threadIdx.x * PER;
        if constexpr (PER == 1) {
            kreg[0] = first < a.max_n ? keys[first] : 0u;
        } else {
#pragma unroll
            for (int e = 0; e < PER; e += 4) {
                uint4 v = make_uint4(0u, 0u, 0u, 0u);  // a row's last piece may reach into its padding
                if (first + e < a.max_n) v = *reinterpret_cast<const uint4*>(keys + first + e);
                kreg[e] = v.x;
                kreg[e + 1] = first + e + 1 < a.max_n ? v.y : 0u;
                kreg[e + 2] = first + e + 2 < a.max_n ? v.z : 0u;
                kreg[e + 3] = first + e + 3 < a.max_n ? v.w : 0u;
            }
        }
        if (topk_direct<NT, PER>(a, kreg, bins, win, wsum, range, s_two)) return;
        if (blockIdx.y != 0) return;  // every workgroup of the row sees the same bins; one searches
        __syncthreads();
        topk_search<NT, PER>(a, kreg, bins, win, wsum, s_two);
    } else {
        const uint32_t none[1] = {0u};
        topk_search<NT, 0>(a, none, bins, win, wsum, s_two);
    }
}

template <int NT, int PER>
inline int launch_topk_as(SortArgs s, int rows, hipStream_t st)
{
    // the search sorts a power of two of entries; the direct path needs room for the bin that crosses place k
    const int most = s.topk < s.max_n ? s.topk : s.max_n;
    int cap = 2;
    while (cap < most) cap <<= 1;
    s.cap = cap;
    // Workgroups per row: one for every NT places.  Each counts the whole row (the keys come from the L2)
    // and orders its share of the places, one entry per thread.
    const int split = PER > 0 ? (int)ucm::ceil_div(most, NT) : 1;
    hipLaunchKernelGGL((topk_kernel<NT, PER>), dim3((unsigned)rows, (unsigned)split), dim3(NT),
                       (size_t)(cap > NT + kCrowd ? cap : NT + kCrowd) * 8, st, s);
    return ucm::launch_status("topk_kernel");
}

// Threads by row length: few where the row fits (a barrier of 4 waves costs less than one of 16: 1000
// candidates as 256 x 4 keys 6.5 us for the whole retrieval call of two short rows, as 1024 x 1 7.1 us;
// 4000 as 512 x 8 and as 1024 x 4 8.3 and 8.5 us), 1024 from where 512 would hold 16 keys each (8000:
// 11.2 us of selection against 8.1 us).
inline int launch_topk(const SortArgs& s, int rows, hipStream_t st)
{
    if (s.max_n <= 256) return launch_topk_as<256, 1>(s, rows, st);
    if (s.max_n <= 1024) return launch_topk_as<256, 4>(s, rows, st);
    if (s.max_n <= 4096) return launch_topk_as<512, 8>(s, rows, st);
    if (s.max_n <= 8192) return launch_topk_as<1024, 8>(s, rows, st);
    if (s.max_n <= 1024 * kMaxRegKeys) return launch_topk_as<1024, kMaxRegKeys>(s, rows, st);
    return launch_topk_as<1024, 0>(s, rows, st);
}

}  // namespace
