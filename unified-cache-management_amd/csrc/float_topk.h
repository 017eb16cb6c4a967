// Selection shared by the float retrieval paths: the k best of a row of fp32 scores in
// descending order, equal scores in list order.  One workgroup per row, or several that order a share of
// its places each; a score travels as an order-preserving 32-bit key that can be turned back into the
// score, so a row is one word per candidate.  Included by the translation units that launch it.
#pragma once

#include <type_traits>

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

// A number that orders like the key, for dividing the rows' range into equal widths.  Both ends lie at half of
// the largest float, so that the range is finite.
__device__ __forceinline__ float key_place(uint32_t k)
{
    const float big = 1.7e38f;
    return fminf(fmaxf(key_score(k), -big), big);  // a NaN, key 1, goes to the lower end
}

// Keys of a row lie at this pitch, whole 64-byte lines: every thread loads its keys as 16-byte pieces.
__host__ __device__ __forceinline__ int64_t key_pitch(int64_t n) { return (n + 15) & ~(int64_t)15; }

struct SortArgs {
    const uint32_t* keys;   // [B] rows of max_n keys, key_pitch(max_n) apart; 16-byte aligned
    const int32_t* idx;     // [B][max_n] what a list position stands for, or null: the position itself
    int max_n, topk, cap;   // cap: entries the search orders in LDS, a power of two
    int32_t* out_idx;       // [B][topk]
    float* out_score;       // [B][topk]
};

// The same as leading arguments of a kernel (see ucm::ArgPair).
#define SORT_ARGS ucm::ArgPair p_in, ucm::ArgPair p_out, ucm::ArgInts n
#define SORT_ARGS_OF(s) ucm::arg_pair((s).keys, (s).idx), ucm::arg_pair((s).out_idx, (s).out_score), ucm::ArgInts{(s).max_n, (s).topk, (s).cap, 0}
__device__ __forceinline__ SortArgs sort_args(SORT_ARGS)
{
    return SortArgs{ucm::arg_ptr<const uint32_t>(p_in.x), ucm::arg_ptr<const int32_t>(p_in.y), n.x, n.y, n.z,
                    ucm::arg_ptr<int32_t>(p_out.x), ucm::arg_ptr<float>(p_out.y)};
}

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

// op over N neighbouring lanes (N = 4, 8 or 16, aligned), in every lane.
template <int N, typename Op>
__device__ __forceinline__ int row_reduce(int v, Op op)
{
    static_assert(N == 4 || N == 8 || N == 16, "lanes of a row");
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, false));   // quad_perm [1,0,3,2]
    v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, false));   // quad_perm [2,3,0,1]
    if (N > 4) v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, false));  // row_half_mirror
    if (N > 8) v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, false));  // row_mirror
    return v;
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
    // a wave's sum a lane, the same in every 16 lanes (words in turn by all waves: 64 instructions instead of 16)
    const int x = wsum[lane % (NT / 64)];
    *total = row_reduce<NT / 64>(x, [](int p, int q) { return p + q; });
    return row_reduce<NT / 64>(lane % (NT / 64) < w ? x : 0, [](int p, int q) { return p + q; }) + inc - v;
}

// What a score is output as: a NaN of one kind, whichever it was.
__device__ __forceinline__ float out_of(uint32_t k) { return k == 1u ? __uint_as_float(0x7fc00000u) : key_score(k); }

// Bins of equal width over the scores between two keys, best first.
template <int BINS>
struct Bins {
    float top, scale;
    __device__ __forceinline__ Bins(uint32_t hi, uint32_t lo) : top(key_place(hi))
    {
        const float width = top - key_place(lo);
        scale = width > 0.0f ? (float)(BINS - 1) / width : 0.0f;
    }
    __device__ __forceinline__ int of(uint32_t k) const
    {
        const float at = (top - key_place(k)) * scale;  // not a number where the scale is infinite: bin 0
        return (int)fminf(fmaxf(at, 0.0f), (float)(BINS - 1));
    }
};

// Direct path.  The row's range of scores is divided into 4 NT bins of equal width, the keys are
// counted per bin, a prefix sum over the bins (best first) says where each bin's entries go, and the
// entries of the bins that start before place k are put there and ranked among the few that share
// their bin.  Where such a bin holds more than kCrowd entries (a few scores far from the rest stretch the
// range: an infinity, one block that holds most of the mass), the entries from the first crowded bin to the
// last are divided again over their own range, up to kAgain times.  Returns false, with nothing written, when
// bins are crowded still (many equal scores, several dense clusters).
// What bounds it is its chain of barriers and LDS round trips, not bytes: one pass over the keys
// replaces the search for the k-th key digit by digit, the compaction and the ordering (4 + 2 + 3
// passes of counting, scanning and placing).  8000 candidates, k = 3000, two rows: 21.0 us for the
// digit search, 8.1 us like this on one workgroup per row, 6.8 us with the places shared by three.  The whole
// call over 128-value rows: even rows 10.9 us, with one infinite score 16.3 (29.8 when the search followed the
// first crowded division).
template <int NT, int PER>
struct Direct {
    static constexpr int kBins = 4 * NT, kAgain = 2;
    const SortArgs& a;
    const uint32_t (&kreg)[PER];
    uint32_t* bins;           // kBins words for every division
    unsigned long long* win;  // NT + kCrowd entries
    int* wsum;
    uint32_t (*range)[NT / 64];
    int* s_int;               // ends of the bins in front of this workgroup's places and of its own; first and last crowded bin;
                              // a bit for every division that has one
    const int b, tid, lane, w;
    // an entry's bin, counted through all divisions, and its place in the bin << 16; in one word where 16 keys
    // leave no registers for two (at 8 keys and less two words are 0.2 us faster)
    static constexpr bool kOneWord = PER > 8;
    uint32_t slot[PER], at[kOneWord ? 1 : PER];
    int n_valid, kk;

    __device__ __forceinline__ int bin(int e) const { return (int)(kOneWord ? slot[e] & 0xffffu : slot[e]); }
    __device__ __forceinline__ int place_of(int e) const { return (int)((kOneWord ? slot[e] : at[e]) >> 16); }
    __device__ __forceinline__ void set(int e, uint32_t bin, uint32_t place)
    {
        slot[e] = kOneWord ? place << 16 | bin : bin;
        if constexpr (!kOneWord) at[e] = place << 16;
    }

    __device__ __forceinline__ Direct(const SortArgs& args, const uint32_t (&k)[PER], uint32_t* lds, int* ws,
                                      uint32_t (*r)[NT / 64], int* si)
        : a(args), kreg(k), bins(lds), win(reinterpret_cast<unsigned long long*>(lds + (1 + kAgain) * kBins)), wsum(ws), range(r),
          s_int(si), b(blockIdx.x), tid(threadIdx.x), lane(threadIdx.x & 63), w(threadIdx.x >> 6)
    {
    }

    // Largest and smallest key of the entries for which in(e), behind a barrier.
    template <class In>
    __device__ __forceinline__ void range_of(In&& in, uint32_t& hi, uint32_t& lo)
    {
        hi = 0u;
        uint32_t l = 0u;  // the smallest as the largest complement
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            if (kreg[e] == 0u || !in(e)) continue;
            hi = kreg[e] > hi ? kreg[e] : hi;
            l = ~kreg[e] > l ? ~kreg[e] : l;
        }
        hi = wave_max(hi);
        l = wave_max(l);
        if (lane == 0) {
            range[0][w] = hi;
            range[1][w] = l;
        }
        __syncthreads();
        auto most = [](int p, int q) { return (int)max((uint32_t)p, (uint32_t)q); };
        hi = (uint32_t)row_reduce<NT / 64>((int)range[0][lane % (NT / 64)], most);
        lo = ~(uint32_t)row_reduce<NT / 64>((int)range[1][lane % (NT / 64)], most);
    }

    // The counts of a division's bins turned into (first place << 16 | entries) words; both fit: a row on this
    // path has at most 16384 candidates.  Behind a barrier, returns whether a bin is crowded.
    __device__ __forceinline__ bool place(int division, int base, uint32_t (&packed)[4])
    {
        uint4* mine = reinterpret_cast<uint4*>(bins + division * kBins) + tid;
        const uint4 c = *mine;
        const uint32_t cnt[4] = {c.x, c.y, c.z, c.w};
        int total, first = base + scan_wg<NT>((int)(c.x + c.y + c.z + c.w), wsum, &total);
        if (division == 0) {
            n_valid = total;
            kk = n_valid < a.topk ? n_valid : a.topk;
        }
        bool crowded = false;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            packed[i] = (uint32_t)first << 16 | cnt[i];
            crowded |= first < kk && cnt[i] > (uint32_t)kCrowd;
            first += (int)cnt[i];
        }
        *mine = make_uint4(packed[0], packed[1], packed[2], packed[3]);
        if (division == 0) mark_ends(packed, 0, 1, 0);
        if (crowded) atomicOr(&s_int[4], 1 << division);
        __syncthreads();
        return s_int[4] >> division & 1;
    }

    // First and last crowded bin of a division, behind a barrier.
    __device__ __forceinline__ void crowd(const uint32_t (&packed)[4], int division, int& f, int& l)
    {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if ((int)(packed[i] >> 16) < kk && (packed[i] & 0xffffu) > (uint32_t)kCrowd) {
                atomicMin(&s_int[2], division * kBins + 4 * tid + i);
                atomicMax(&s_int[3], division * kBins + 4 * tid + i);
            }
        }
        __syncthreads();
        f = s_int[2];
        l = s_int[3];
    }

    // This workgroup's share of the places: the entries of the bins that start in [lo_at, hi_at).
    __device__ __forceinline__ void share(int& lo_at, int& hi_at) const
    {
        const int n = (kk + (int)gridDim.y - 1) / (int)gridDim.y;
        lo_at = (int)blockIdx.y * n < kk ? (int)blockIdx.y * n : kk;
        hi_at = lo_at + n < kk ? lo_at + n : kk;
    }

    // Where the bins end that hold the places in front of lo_at and of hi_at: one thread has each.  b0 .. b1: bins
    // that are divided again.
    __device__ __forceinline__ void mark_ends(const uint32_t (&packed)[4], int division, int b0, int b1) const
    {
        int lo_at, hi_at;
        share(lo_at, hi_at);
        const int from = (int)(packed[0] >> 16), to = (int)(packed[3] >> 16) + (int)(packed[3] & 0xffffu);
        if (!((from < lo_at && lo_at <= to) || (from < hi_at && hi_at <= to))) return;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int j = division * kBins + 4 * tid + i;
            if (j >= b0 && j <= b1) continue;
            const int first = (int)(packed[i] >> 16), end = first + (int)(packed[i] & 0xffffu);
            if (first < lo_at && lo_at <= end) s_int[0] = end;
            if (first < hi_at && hi_at <= end) s_int[1] = end;
        }
    }

    // Entries to their bins' places, ranked there, and out.  bin_of(key): the entry's bin.
    template <class BinOf>
    __device__ __forceinline__ void finish(BinOf&& bin_of) const
    {
        int lo_at, hi_at;
        share(lo_at, hi_at);
        int at_bin[PER];  // all read in front of the first write (a key that is none has some bin, too)
#pragma unroll
        for (int e = 0; e < PER; ++e) at_bin[e] = (int)(bins[bin(e)] >> 16);
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            const int f = at_bin[e];
            if (kreg[e] != 0u && f >= lo_at && f < hi_at) win[f - lo_at + place_of(e)] = ((unsigned long long)kreg[e] << 32) | (uint32_t)(~(uint32_t)(tid * PER + e));
        }
        __syncthreads();
        const int end = s_int[1];
        for (int i = s_int[0] + tid; i < end; i += NT) {
            const unsigned long long x = win[i - lo_at];
            const uint32_t k = (uint32_t)(x >> 32);
            const int pos = (int)(~(uint32_t)x);
            const int32_t id = a.idx ? a.idx[(int64_t)b * a.max_n + pos] : pos;
            const uint32_t p = bins[bin_of(k)];
            const int f = (int)(p >> 16), n = (int)(p & 0xffffu);
            int rank = f;  // entries of the bin that go before this one come first
            for (int j = 0; j < n; j += 4) {  // four a round trip, places past the bin's last repeat it
                unsigned long long o[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) o[u] = win[f - lo_at + (j + u < n ? j + u : n - 1)];
#pragma unroll
                for (int u = 0; u < 4; ++u) rank += j + u < n && o[u] > x;
            }
            if (rank < kk) {
                a.out_idx[(int64_t)b * a.topk + rank] = id;
                a.out_score[(int64_t)b * a.topk + rank] = out_of(k);
            }
        }
        for (int t = kk + (int)blockIdx.y * NT + tid; t < a.topk; t += NT * (int)gridDim.y) {
            a.out_idx[(int64_t)b * a.topk + t] = -1;
            a.out_score[(int64_t)b * a.topk + t] = 0.0f;
        }
    }

    __device__ __forceinline__ bool run()
    {
        reinterpret_cast<uint4*>(bins)[tid] = make_uint4(0u, 0u, 0u, 0u);
        if (tid < 5) s_int[tid] = tid == 2 ? (1 + kAgain) * kBins : (tid == 3 ? -1 : 0);
        uint32_t hi, lo;
        range_of([](int) { return true; }, hi, lo);
        const Bins<kBins> whole(hi, lo);
        // 64 lanes adding to one LDS word serialise: where the wave's first keys share a bin, so may the others,
        // and one lane adds for all that have its own (a row that one infinite score crowds into a bin: 4 us less)
#pragma unroll
        for (int e = 0; e < PER; ++e) set(e, (uint32_t)whole.of(kreg[e]), 0u);
        const int bin0 = __builtin_amdgcn_readfirstlane(bin(0));
        if (__ballot(kreg[0] != 0u && bin(0) == bin0) == ~0ull) {
            const unsigned long long before = (1ull << lane) - 1;
#pragma unroll
            for (int e = 0; e < PER; ++e) {
                const unsigned long long same = __ballot(kreg[e] != 0u && bin(e) == bin0);
                uint32_t base = 0u;
                if (lane == 0) base = atomicAdd(&bins[bin0], (uint32_t)__popcll(same));
                base = __builtin_amdgcn_readfirstlane(base);
                if (same >> lane & 1) set(e, (uint32_t)bin(e), base + (uint32_t)__popcll(same & before));
                else if (kreg[e] != 0u) set(e, (uint32_t)bin(e), atomicAdd(&bins[bin(e)], 1u));
            }
        } else {
            bool all = true;
#pragma unroll
            for (int e = 0; e < PER; ++e) all &= kreg[e] != 0u;
            if (__ballot(all) == ~0ull) {  // no test between the additions: they are one round trip
                uint32_t place[PER];
#pragma unroll
                for (int e = 0; e < PER; ++e) place[e] = atomicAdd(&bins[bin(e)], 1u);
#pragma unroll
                for (int e = 0; e < PER; ++e) set(e, (uint32_t)bin(e), place[e]);
            } else {
#pragma unroll
                for (int e = 0; e < PER; ++e)
                    if (kreg[e] != 0u) set(e, (uint32_t)bin(e), atomicAdd(&bins[bin(e)], 1u));
            }
        }
        __syncthreads();
        uint32_t packed[4];
        if (place(0, 0, packed)) return run_again(whole, packed);
        finish([&](uint32_t k) { return whole.of(k); });
        return true;
    }

    __device__ __forceinline__ bool run_again(const Bins<kBins>& whole, const uint32_t (&packed0)[4])
    {
        uint32_t packed[1 + kAgain][4];
        int b0[1 + kAgain], b1[1 + kAgain];  // per division: its bins that are divided again
        Bins<kBins> part[1 + kAgain] = {whole, whole, whole};
        static_assert(kAgain == 2, "");
#pragma unroll
        for (int i = 0; i < 4; ++i) packed[0][i] = packed0[i];
        bool crowded = true;
#pragma unroll
        for (int d = 1; d <= kAgain; ++d) {
            b0[d] = (1 + kAgain) * kBins;
            b1[d] = -1;
            if (!crowded) continue;
            int f, l;
            crowd(packed[d - 1], d - 1, f, l);
            b0[d - 1] = f;
            b1[d - 1] = l;
            reinterpret_cast<uint4*>(bins + d * kBins)[tid] = make_uint4(0u, 0u, 0u, 0u);
            uint32_t hi, lo;
            range_of([&](int e) { return bin(e) >= f && bin(e) <= l; }, hi, lo);
            if (hi == lo) return false;  // ties
            part[d] = Bins<kBins>(hi, lo);
            // every thread has read the last two: range_of() has a barrier
            if (tid < 4) s_int[tid] = tid == 2 ? (1 + kAgain) * kBins : (tid == 3 ? -1 : 0);
#pragma unroll
            for (int e = 0; e < PER; ++e) {
                if (kreg[e] == 0u || bin(e) < f || bin(e) > l) continue;
                const uint32_t j = (uint32_t)(d * kBins + part[d].of(kreg[e]));
                set(e, j, atomicAdd(&bins[j], 1u));
            }
            __syncthreads();
            crowded = place(d, (int)(bins[f] >> 16), packed[d]);
        }
        if (crowded) return false;
#pragma unroll
        for (int d = 0; d <= kAgain; ++d)
            if (d == 0 || b0[d - 1] <= b1[d - 1]) mark_ends(packed[d], d, b0[d], b1[d]);
        finish([&](uint32_t k) {
            int j = whole.of(k);
#pragma unroll
            for (int d = 1; d <= kAgain; ++d)
                if (j >= b0[d - 1] && j <= b1[d - 1]) j = d * kBins + part[d].of(k);
            return j;
        });
        return true;
    }
};

// Any row.  Radix passes of 10 or 11 bits find the k-th largest key, winners go to LDS at slots from one
// prefix sum (keys above the threshold, then the ties in list order), and the (key, position) pairs above the
// threshold are ordered: equal-width buckets over (threshold, largest key], or bitonic networks and pairwise
// merges where a bucket is crowded.  PER = 0: keys are re-read from memory in every phase (rows longer than
// the registers hold).  Where the direct path was tried in vain, three passes instead of four of 8 bits, no
// ordering of the ties and no second count of the candidates pay for it: two rows of 4000 candidates, k = 1200,
// all scores equal 16.5 us for the call (34.4 with four passes and no attempt in front), four different ones
// 35.5 (35.9).
// lds: 4 NT words, then the winners (a.cap of 8 bytes).  n_valid: candidates of the row, -1 = not known.
template <int NT, int PER>
__device__ void topk_search(const SortArgs& a, const uint32_t (&kreg)[PER ? PER : 1], uint32_t* lds, int* wsum, int* s_two,
                            int n_valid)
{
    constexpr bool REG = PER > 0;
    constexpr int kBuckets = NT;  // one per thread
    constexpr int kDigitBits = NT >= 512 ? 11 : 10, kPerThread = (1 << kDigitBits) / NT;
    static_assert(kPerThread >= 1 && (1 << kDigitBits) <= 4 * NT, "");
    unsigned long long* win = reinterpret_cast<unsigned long long*>(lds + 4 * NT);
    int* hist = reinterpret_cast<int*>(lds);
    int* bcount = reinterpret_cast<int*>(lds);      // kBuckets each, after the search
    int* bfill = bcount + kBuckets;
    int* bbase = bfill + kBuckets;
    const int b = blockIdx.x;
    const uint32_t* keys = a.keys + b * key_pitch(a.max_n);
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

    if (n_valid < 0) {
        int mine = 0;
        for_chunks([&](int, uint32_t k) { mine += k != 0u; });
        (void)scan_wg<NT>(mine, wsum, &n_valid);
    }
    const int kk = n_valid < a.topk ? n_valid : a.topk;

    // ---- radix search for the kk-th largest key among the candidates ----
    uint32_t prefix = 0, mask = 0;
    int need = kk;
    for (int below = 32; below > 0 && kk > 0;) {  // bits not known yet
        const int bits = below < kDigitBits ? below : kDigitBits, shift = below - bits, last = (1 << bits) - 1;
#pragma unroll
        for (int j = 0; j < kPerThread; ++j) hist[tid + j * NT] = 0;
        __syncthreads();
        for_chunks([&](int, uint32_t k) {
            const bool in = k != 0u && (k & mask) == prefix;
            const int d = (k >> shift) & last;
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
        // digits in descending order, kPerThread to a thread: the chosen digit is where the running
        // count first reaches `need`
        int cnt[kPerThread], sum = 0, all;
#pragma unroll
        for (int j = 0; j < kPerThread; ++j) {
            const int d = last - (tid * kPerThread + j);
            cnt[j] = d >= 0 ? hist[d] : 0;
            sum += cnt[j];
        }
        int before = scan_wg<NT>(sum, wsum, &all);
#pragma unroll
        for (int j = 0; j < kPerThread; ++j) {
            if (before < need && before + cnt[j] >= need) {
                s_two[0] = last - (tid * kPerThread + j);
                s_two[1] = need - before;  // still to take among keys with this digit
            }
            before += cnt[j];
        }
        __syncthreads();
        prefix |= (uint32_t)s_two[0] << shift;
        mask |= (uint32_t)last << shift;
        need = s_two[1];
        below = shift;
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

    // ---- order the winners above the threshold, descending: larger key first, then smaller position (the
    //      ties behind them are in list order already) ----
    // Their keys lie in (thr, kmax]; equal-width buckets over that range (descending), a prefix sum over the
    // bucket counts, every winner dropped into its bucket, then ranked among the few entries that share it.
    if (n_gt > 1) {
        constexpr int kPer = REG && NT * PER < kMaxTopk ? PER : kMaxTopk / NT;  // entries per thread at the largest cap
        uint32_t kmax = 0u;
        unsigned long long x[kPer];
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
            const int i = tid + e * NT;
            x[e] = i < n_gt ? win[i] : 0ull;
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
            if (i < n_gt) {
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
            int cap = 2;  // entries of the networks: the ties that fall inside stay behind all others, in their order
            while (cap < n_gt) cap <<= 1;
            const int seg = cap < 256 ? cap : 256;
            for (int size = 2; size <= seg; size <<= 1) {
                for (int stride = size >> 1; stride > 0; stride >>= 1) {
                    for (int t = tid; t < cap / 2; t += NT) {
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
            for (int run = seg; run < cap; run <<= 1) {
                int dst[kPer];
                const int sh = __builtin_ctz(run);
#pragma unroll
                for (int e = 0; e < kPer; ++e) {
                    const int i = tid + e * NT;
                    dst[e] = -1;
                    if (i < cap) {
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
    }

    for (int t = tid; t < a.topk; t += NT) {
        int32_t oi = -1;
        float os = 0.0f;
        if (t < kk) {
            const int pos = (int)(~(uint32_t)(win[t] & 0xffffffffull));
            const uint32_t k = (uint32_t)(win[t] >> 32);
            oi = a.idx ? a.idx[(int64_t)b * a.max_n + pos] : pos;
            os = out_of(k);
        }
        a.out_idx[(int64_t)b * a.topk + t] = oi;
        a.out_score[(int64_t)b * a.topk + t] = os;
    }
}

// Short rows: every candidate counts those that come before it in the output order (larger key, or equal key
// and earlier position) and writes itself at that rank.  Its time does not depend on the values.  A workgroup
// ranks 64 candidates; its waves compare them with every so many 64 entries of the row.  grid = (rows, ceil(max_n / 64)).
template <int WAVES>
struct RankShared {
    __attribute__((aligned(16))) uint32_t key[WAVES][64];
    uint32_t part[WAVES][64];  // ranks among a wave's entries, and in the upper half how many of them there are
};

// mine: the lane's candidate of the workgroup; first: of the wave's first 64, where has_first says that it is known.
// UNROLL: reads of four keys to a step of the loop over a wave's 64.
template <int WAVES, int UNROLL, typename Key>
__device__ __forceinline__ void rank_places(const SortArgs& a, int waves, uint32_t mine, uint32_t first, bool has_first,
                                            Key key_of, RankShared<WAVES>& sh)
{
    const int b = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6, mine_at = blockIdx.y;
    const int pos = mine_at * 64 + lane;
    const int32_t id = w == 0 && a.idx && pos < a.max_n ? a.idx[(int64_t)b * a.max_n + pos] : pos;
    int rank = 0, have = 0;
    for (int piece = w; piece * 64 < a.max_n; piece += waves) {
        const uint32_t k = has_first && piece == w ? first : key_of(piece * 64 + lane);
        have += __popcll(__ballot(k != 0u));
        // A wave's keys go round by way of LDS, four to a read that all lanes share.
        sh.key[w][lane] = k;
        __builtin_amdgcn_wave_barrier();
        const uint4* all = reinterpret_cast<const uint4*>(sh.key[w]);
        auto count = [&](auto own_) {
#pragma unroll UNROLL
            for (int j = 0; j < 64; j += 4) {
                const uint4 o4 = all[j / 4];
                const uint32_t o[4] = {o4.x, o4.y, o4.z, o4.w};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if constexpr (decltype(own_)::value) rank += o[i] > mine || (o[i] == mine && j + i < lane);
                    // equal keys come first where they lie in front: o >= mine is o > mine - 1 (mine is 0 for nothing only)
                    else rank += o[i] > mine - (piece < mine_at ? 1u : 0u);
                }
            }
        };
        if (piece == mine_at) count(std::true_type{});
        else count(std::false_type{});
        __builtin_amdgcn_wave_barrier();
    }
    sh.part[w][lane] = (uint32_t)rank | (uint32_t)have << 16;
    __syncthreads();
    if (w != 0) return;
    uint32_t sum = 0;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) {
        const uint32_t p = sh.part[i][lane];
        sum += i < waves ? p : 0u;
    }
    rank = (int)(sum & 0xffffu);
    const int n_valid = (int)(sum >> 16);
    if (mine != 0u && rank < a.topk) {
        a.out_idx[(int64_t)b * a.topk + rank] = id;
        a.out_score[(int64_t)b * a.topk + rank] = out_of(mine);
    }
    for (int t = n_valid + pos; t < a.topk; t += 64 * (int)gridDim.y) {
        a.out_idx[(int64_t)b * a.topk + t] = -1;
        a.out_score[(int64_t)b * a.topk + t] = 0.0f;
    }
}

// All 64 keys in a row, as a wave has up to two pieces: 8 and 32 rows of 400 candidates 4.4 and 4.5 us, eight keys to a step 4.7 and 4.9,
// lane by lane through a scalar register 4.5 and 4.55 (one row of 253: 3.3, 3.3 and 3.5).
constexpr int kRankRow = 512;
__global__ __launch_bounds__(256) void topk_rank_kernel(SORT_ARGS)
{
    __shared__ RankShared<4> sh;
    const SortArgs a = sort_args(p_in, p_out, n);
    const uint32_t* keys = a.keys + blockIdx.x * key_pitch(a.max_n);
    const int pos = blockIdx.y * 64 + (threadIdx.x & 63);
    const uint32_t mine = pos < a.max_n ? keys[pos] : 0u;
    rank_places<4, 16>(a, 4, mine, 0u, false, [&](int at) { return at < a.max_n ? keys[at] : 0u; }, sh);
}

// The same for one row of up to kRankSums candidates whose scores are still in n_sums parts, which every workgroup
// adds by itself, in the same order.  A wave for every 64 candidates up to sixteen: the parts of a wave's 64 and those
// of the workgroup's own 64 are one round trip (253 candidates of 16 parts: 3.9 us, with its arguments read from memory 4.7, requested a
// few at a time 5.0; 1024 of them 3 us less than in four waves with a branch at every part).  Eight keys to a step of the ranking's
// loop: code is fetched anew by every launch, and sixteen waves in straight line wait for it (253 candidates 3.9 and 4.4 us, 1024: 5.3 and 6.2).
constexpr int kRankSums = 2048;
__global__ __launch_bounds__(1024) void topk_rank_sums_kernel(SORT_ARGS)
{
    __shared__ RankShared<16> sh;
    SortArgs a = sort_args(p_in, p_out, n);
    const float* const sums = reinterpret_cast<const float*>(a.keys);
    const int max_n = n.x, n_sums = n.z;
    a.idx = nullptr;
    auto keys_of = [&](auto n_, const int (&at)[decltype(n_)::value], uint32_t (&key)[decltype(n_)::value]) {
        constexpr int N = decltype(n_)::value;
        double s[N] = {};  // sixteen parts one after the other in 32 bits were the largest error of a block's score
        uint32_t off[N];
#pragma unroll
        for (int n = 0; n < N; ++n) off[n] = at[n] < max_n ? at[n] : max_n - 1;
        for (int i = 0; i < n_sums; i += 16) {
            float v[N][16];
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float* p = sums + (int64_t)(i + e < n_sums ? i + e : 0) * max_n;
#pragma unroll
                for (int n = 0; n < N; ++n) v[n][e] = p[off[n]];
            }
            __builtin_amdgcn_sched_barrier(0);  // all requested before the first is waited for
#pragma unroll
            for (int e = 0; e < 16; ++e)
#pragma unroll
                for (int n = 0; n < N; ++n) s[n] += i + e < n_sums ? (double)v[n][e] : 0.0;
        }
#pragma unroll
        for (int n = 0; n < N; ++n) key[n] = at[n] < max_n ? score_key((float)s[n]) : 0u;
    };
    const int lane = threadIdx.x & 63;
    const int at[2] = {(int)blockIdx.y * 64 + lane, (int)threadIdx.x};
    uint32_t key[2];
    keys_of(std::integral_constant<int, 2>{}, at, key);
    rank_places<16, 2>(a, blockDim.x / 64, key[0], key[1], true, [&](int p) {
        const int one[1] = {p};
        uint32_t k[1];
        keys_of(std::integral_constant<int, 1>{}, one, k);
        return k[0];
    }, sh);
}

// LDS of topk_kernel: bins and winners, as the two paths lay them out.
constexpr size_t direct_lds(int nt) { return (size_t)nt * 48 + (size_t)(nt + kCrowd) * 8; }
constexpr size_t search_lds(int nt, int cap) { return (size_t)nt * 16 + (size_t)cap * 8; }

// grid = (rows, workgroups per row).  Thread t holds list positions t * PER ..
// t * PER + PER - 1 (consecutive, so that one prefix sum over per-thread counts orders the list).
template <int NT, int PER>
__global__ __launch_bounds__(NT) void topk_kernel(SORT_ARGS)
{
    const SortArgs a = sort_args(p_in, p_out, n);
    extern __shared__ __align__(16) uint32_t lds[];
    __shared__ int wsum[NT / 64];
    __shared__ uint32_t range[2][NT / 64];
    __shared__ int s_int[5];
    if constexpr (PER > 0) {
        static_assert(PER % 4 == 0, "16-byte loads");
        uint32_t kreg[PER];
        const uint32_t* keys = a.keys + blockIdx.x * key_pitch(a.max_n);
        const int first = threadIdx.x * PER;
#pragma unroll
        for (int e = 0; e < PER; e += 4) {
            uint4 v = make_uint4(0u, 0u, 0u, 0u);  // a row's last piece may reach into its padding
            if (first + e < a.max_n) v = *reinterpret_cast<const uint4*>(keys + first + e);
            kreg[e] = v.x;
            kreg[e + 1] = first + e + 1 < a.max_n ? v.y : 0u;
            kreg[e + 2] = first + e + 2 < a.max_n ? v.z : 0u;
            kreg[e + 3] = first + e + 3 < a.max_n ? v.w : 0u;
        }
        Direct<NT, PER> direct(a, kreg, lds, wsum, range, s_int);
        if (direct.run()) return;
        if (blockIdx.y != 0) return;  // every workgroup of the row sees the same bins; one searches
        __syncthreads();
        topk_search<NT, PER>(a, kreg, lds, wsum, s_int, direct.n_valid);
    } else {
        const uint32_t none[1] = {0u};
        topk_search<NT, 0>(a, none, lds, wsum, s_int, -1);
    }
}

template <int NT, int PER>
inline int launch_topk_as(SortArgs s, int rows, hipStream_t st)
{
    // the search sorts a power of two of entries
    const int most = s.topk < s.max_n ? s.topk : s.max_n;
    int cap = 2;
    while (cap < most) cap <<= 1;
    s.cap = cap;
    // Workgroups per row: one for every NT places.  Each counts the whole row (the keys come from the L2)
    // and orders its share of the places, one entry per thread.
    const int split = PER > 0 ? (int)ucm::ceil_div(most, NT) : 1;
    const size_t need = search_lds(NT, cap), direct = PER > 0 ? direct_lds(NT) : 0;
    static_assert(search_lds(NT, kMaxTopk) + 512 <= 64 * 1024 && direct_lds(NT) + 512 <= 64 * 1024, "");
    hipLaunchKernelGGL((topk_kernel<NT, PER>), dim3((unsigned)rows, (unsigned)split), dim3(NT), need > direct ? need : direct, st, SORT_ARGS_OF(s));
    return ucm::launch_status("topk_kernel");
}

// One row of up to kRankSums candidates whose scores are in n_sums parts, [n_sums][s.max_n].
inline int launch_rank_sums(const SortArgs& s, const float* sums, int n_sums, hipStream_t st)
{
    const unsigned pieces = (unsigned)ucm::ceil_div(s.max_n, 64);
    hipLaunchKernelGGL(topk_rank_sums_kernel, dim3(1, pieces), dim3(64 * (pieces < 16 ? pieces : 16)), 0, st,
                       ucm::arg_pair(sums, nullptr), ucm::arg_pair(s.out_idx, s.out_score), ucm::ArgInts{s.max_n, s.topk, n_sums, 0});
    return ucm::launch_status("topk_rank_sums_kernel");
}

// Rows of up to 512 candidates are ranked: as fast as the direct path on an even row (two rows, whole call: 253
// candidates 6.0 against 5.8 us, 400: 6.7 and 6.4, 700: 7.5 and 6.9) and faster on one that crowds (400: 8.9 with a
// second division, 11 to 18 with the search).
// Threads by row length: few where the row fits (a barrier of 4 waves costs less than one of 16: 1000
// candidates as 256 x 4 keys 6.5 us for the whole retrieval call of two short rows, as 1024 x 1 7.1 us;
// 4000 as 512 x 8 and as 1024 x 4 8.3 and 8.5 us), 1024 from where 512 would hold 16 keys each (8000:
// 11.2 us of selection against 8.1 us).
inline int launch_topk(const SortArgs& s, int rows, hipStream_t st)
{
    if (s.max_n <= kRankRow) {
        hipLaunchKernelGGL(topk_rank_kernel, dim3((unsigned)rows, (unsigned)ucm::ceil_div(s.max_n, 64)), dim3(256), 0, st, SORT_ARGS_OF(s));
        return ucm::launch_status("topk_rank_kernel");
    }
    if (s.max_n <= 1024) return launch_topk_as<256, 4>(s, rows, st);
    if (s.max_n <= 4096) return launch_topk_as<512, 8>(s, rows, st);
    if (s.max_n <= 8192) return launch_topk_as<1024, 8>(s, rows, st);
    if (s.max_n <= 1024 * kMaxRegKeys) return launch_topk_as<1024, kMaxRegKeys>(s, rows, st);
    return launch_topk_as<1024, 0>(s, rows, st);
}

}  // namespace
