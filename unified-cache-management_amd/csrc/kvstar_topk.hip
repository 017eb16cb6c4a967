// KVStar block retrieval for gfx950: attention-probability mass per KV block, then top-k.
//
// GPU counterpart of the reference's CPU kernel
// (ucm/sparse/kvstar/retrieve/core/domain/retrieve_task/simd_compute_kernel.cpp:816-985, the
// scalar form; its NEON / AVX forms compute the same quantities in other summation orders):
//   1. optional channel pruning of the queries: q'[x, H, j] = q[x, H, pruned_index[H / g, j]];
//   2. scores[x, H, s] = q'[x, H, :] . k[s, H / g, :] over the S = n_blocks * M block
//      representatives, fp16 inputs, fp32 accumulation;
//   3. softmax over s for every (x, H) (left unnormalised when the sum of exponentials is
//      <= 1e-9, as the reference does);
//   4. block score[n] = sum over x, H and the M representatives of block n;
//   5. the topk blocks by descending score.
// Two ways, by the shape of the blocks; the [X Hq, S] score matrix is stored by neither (writing it and reading it
// back twice moved seven times the bytes of the keys themselves).
//   * Blocks of 16, 32 or up to four times 64 representatives of 32, 64 or 128 channels, up to kRankSums of them:
//     kvstar_unit_kernel (q.k on the matrix cores; maximum and sum of exponentials of every row and block),
//     kvstar_merge_kernel (probabilities of them, summed over sixteen rows) and the ranking, which adds the last sums.
//   * Everything else: kvstar_stats_kernel (maximum and sum of exponentials of every row over one chunk of the
//     representatives), kvstar_mass_kernel (the chunks' pairs merged, q.k once more, probabilities summed over rows
//     and a block's representatives) and the shared top-k selection.
// 8 query tokens x 32 heads, 253 blocks x 64 representatives, 32 channels: 13.0 to 13.3 us (6.2, 3.9 and 3.9 of the three
// kernels: launches and round trips; the products and exponentials are about 1.5), 18.8 the second way
// (7.5, 9.0, 3.7); 1024 blocks, 128 channels: 36.1 and 70.4, the second way reads the keys twice.
// Error against 64 bits at that shape 3.3e-8 of the scores' 2-norm (the second way 4.8e-8), over 34 others of like
// values (1 to 16 tokens, 24 to 1000 blocks of 16 to 256, 32 to 128 channels) 2.8e-8 to 3.8e-7 (3.5e-8 to 3.9e-7).
// Sums are taken in a different order than the reference's loops, the same one on every call (no
// atomics); the tolerance is stated where the results are compared.  Equal scores come out in
// ascending block order (the reference's heap pops them in descending block order).
#include <hip/hip_fp16.h>

#include <type_traits>

#include "common.h"
#include "exp_sum.h"
#include "float_topk.h"

namespace {

constexpr int kThreads = 512;       // both kernels: eight waves
constexpr int kAnyDim = 0;          // KS of the statistics kernel for other dimensions than 32, 64 and 128, up to
constexpr int kAnyDimMost = 512;    // this (32 rows in LDS), and
constexpr int kPacked = -1;         // for those above it, whose query rows kvstar_pack_kernel has gathered
constexpr int stat_items(int ks) { return ks > 0 ? 2 : 1; }  // row tiles a workgroup of it serves
constexpr int kEarly = 8;           // k-steps that kernels for any dimension request ahead of their other work,
constexpr int kEarlyMost = 256;     // in rows up to this (512 channels, 16 representatives: 0.8 us more with it)
constexpr int kLongDim = 128;       // above it loads take more of both kernels' time than the statistics' merging
constexpr int kMaxChunks = 64;      // partial statistics per row
constexpr int kLeastTiles = 4;      // tiles of a chunk
constexpr int kMassRows = 2048;     // rows whose statistics the mass kernel holds in LDS at a time
constexpr int kMassGroups = 512;    // its workgroups at most
constexpr int kMergeRows = 16;      // query rows of a workgroup of the merge kernel
constexpr int kUnitGroups = 512;    // workgroups of the unit kernel at most
constexpr int64_t kUnitBytes = 64 << 20;  // its pairs at most

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Largest score of a part of a row and the sum of exp(score - m) over it; (-inf, 0) where nothing was seen.
// Scores reach 4.4e12 for finite inputs (1024 channels), where fp32 steps are 2^18: only the difference of
// two scores, which is exact when they are close, is ever an exponent.
struct Stat {
    float m;
    float s;
};

// The X * g query rows of a KV head are cut into tiles of 32; item = h * tiles_q + tile.
struct KvArgs {
    const _Float16* q;      // [X, Hq, d_orig]
    const _Float16* k;      // [S, Hkv, d]
    const int64_t* pruned;  // [Hkv, d] or null
    int X, Hq, Hkv, g, d_orig, d;
    int64_t S;
    int n_blocks, M;
    int tiles_q, items;     // row tiles per KV head, and of all heads
    int tiles_k, per_chunk; // tiles of 32 representatives: all, and per chunk of the statistics kernel
    int chunks;
    int dp;                 // d in whole steps of 16 channels
    _Float16* qp;           // [items][32][dp] query rows, channels pruned, zeros behind the last row and channel
    Stat* part;             // [chunks][items * 32] sum of exponentials over a chunk, or [units][items * 32] over a unit
    uint32_t* keys;         // [n_blocks]
    float* sums;            // [items * 32 / kMergeRows][units] probabilities of a unit, summed over so many rows
    int units;              // a unit is a block, where all of a row's fit (0: chunks instead)
    int group_blocks;       // blocks a workgroup of the mass kernel handles together
    int groups;
};

typedef _Float16 f16x8u __attribute__((ext_vector_type(8), aligned(2)));

// Channels c .. c + 7 of a representative's row, zeros past d.
__device__ __forceinline__ f16x8 load_k(const _Float16* row, int c, int d)
{
    f16x8 v = {0};
    if (c + 8 <= d) {
        v = *reinterpret_cast<const f16x8u*>(row + c);
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = c + i < d ? row[c + i] : (_Float16)0;
    }
    return v;
}

// The query row of place r of an item: KV head h's row rr = x * g + gg belongs to query head h * g + gg.
struct QRow {
    const _Float16* row;
    const int64_t* pruned;  // the KV head's channels, or null
    bool ok;
};

__device__ __forceinline__ QRow q_row(const KvArgs& a, int item, int r)
{
    const int h = a.tiles_q == 1 ? item : item / a.tiles_q;
    const int rr = (item - h * a.tiles_q) * 32 + r;
    const int x = (a.g & (a.g - 1)) == 0 ? rr >> __builtin_ctz(a.g) : rr / a.g;  // (a division is forty instructions)
    QRow q;
    q.ok = item < a.items && rr < a.X * a.g;
    q.row = a.q + ((int64_t)(q.ok ? x : 0) * a.Hq + (q.ok ? h * a.g + rr - x * a.g : 0)) * a.d_orig;
    q.pruned = a.pruned ? a.pruned + (int64_t)(q.ok ? h : 0) * a.d : nullptr;
    return q;
}

// Channel j of a query row; an index outside the row is moved to its ends.
__device__ __forceinline__ int64_t q_channel(const QRow& q, int j, int d_orig)
{
    const int64_t src = q.pruned ? q.pruned[j] : j;
    return src < 0 ? 0 : (src >= d_orig ? d_orig - 1 : src);
}

// Channels c .. c + 7 of a query row, zeros past d and for a row that does not exist.
__device__ __forceinline__ f16x8 load_q(const QRow& q, int c, int d, int d_orig)
{
    f16x8 v;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = q.ok && c + i < d ? q.row[q_channel(q, c + i, d_orig)] : (_Float16)0;
    return v;
}

constexpr float kLog2e = 1.44269502f, kLog2eLow = 1.92596303e-8f;  // log2(e) in two pieces

// exp(x) for x far from overflow (here x <= 0 but for rounding): 2^(x log2 e) with log2 e in two pieces and the
// product's rounding error carried along (Dekker's exact product, by a fused multiply-add), whole and fractional
// part of the exponent taken apart so that results down to the smallest denormal come out.  A NaN stays one.
__device__ __forceinline__ float exp_small(float x)
{
    x = __builtin_elementwise_maximum(x, -200.0f);  // also minus infinity; the result is 0 either way
    const float t = x * kLog2e;
    const float n = __builtin_rintf(t);
    const float r = __builtin_fmaf(x, kLog2eLow, __builtin_fmaf(x, kLog2e, -t));
    return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f((t - n) + r), (int)n);
}

// What a part's maximum is measured from: 0 where the largest one is minus infinity, whose exponentials are 0.
__device__ __forceinline__ float stat_base(float m) { return m == -INFINITY ? 0.0f : m; }

// The factor exp(x) of a part whose maximum lies x <= 0 off the largest.  Rounding the exponent moves it by
// |x| 2^-24 of itself, at most 2^-25 of the row's sum, which holds a term of 1: that error need not be carried
// as in exp_small (1.1 us more at the example's shape), only log2(e)'s own, which has the same sign in every part.
__device__ __forceinline__ float part_weight(float x)
{
    return __builtin_amdgcn_exp2f(__builtin_fmaf(x, kLog2e, x * kLog2eLow));
}

// `st` and the first `count` of the parts v.
template <int N>
__device__ __forceinline__ Stat merge(Stat st, const Stat (&v)[N], int count = N)
{
    float m = st.m;
#pragma unroll
    for (int i = 0; i < N; ++i) m = fmaxf(m, i < count ? v[i].m : -INFINITY);
    const float base = stat_base(m);
    float sum = st.s * part_weight(st.m - base);
#pragma unroll
    for (int i = 0; i < N; ++i) sum += i < count ? v[i].s * part_weight(v[i].m - base) : 0.0f;
    return Stat{m, sum};
}

// Two parts of a sum that is not a row's but a block's, where its own size is what is asked for: an exact weight.
__device__ __forceinline__ Stat join(Stat a, Stat b)
{
    const float m = fmaxf(a.m, b.m);
    const float w = exp_small(fminf(a.m, b.m) - stat_base(m));
    return Stat{m, a.m < b.m ? a.s * w + b.s : a.s + b.s * w};
}

// Any head dimension: U tiles of representatives against a row tile, up to eight k-steps' loads in flight (16
// bytes each, representatives of an odd dimension from any even address).  The steps are added in ascending
// order, as where their number is known: both kernels get the same score to the last bit.  QA: the query rows
// are the A operand.  c: the first channel to add.
template <bool QA, int U>
__device__ __forceinline__ void dots_any(const _Float16* qrow, const _Float16* const (&row)[U], int kb, int c, int d,
                                         f32x16 (&acc)[U])
{
    auto mul = [&](const f16x8& q, const f16x8& k, f32x16& c) {
        c = QA ? __builtin_amdgcn_mfma_f32_32x32x16_f16(q, k, c, 0, 0, 0) : __builtin_amdgcn_mfma_f32_32x32x16_f16(k, q, c, 0, 0, 0);
    };
    auto steps = [&](int c, auto n_) {
        constexpr int N = decltype(n_)::value;
        f16x8 q[N], k[U][N];
#pragma unroll
        for (int u = 0; u < U; ++u)  // a row's pieces one after the other: four of them share a cache line
#pragma unroll
            for (int i = 0; i < N; ++i) k[u][i] = *reinterpret_cast<const f16x8u*>(row[u] + c + i * 16 + kb);
#pragma unroll
        for (int i = 0; i < N; ++i) q[i] = *reinterpret_cast<const f16x8*>(qrow + c + i * 16 + kb);
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int u = 0; u < U; ++u) mul(q[i], k[u][i], acc[u]);
    };
    for (; c + 128 <= d; c += 128) steps(c, std::integral_constant<int, 8>{});
    if (c + 64 <= d) {
        steps(c, std::integral_constant<int, 4>{});
        c += 64;
    }
    if (c + 32 <= d) {
        steps(c, std::integral_constant<int, 2>{});
        c += 32;
    }
    if (c + 16 <= d) {
        steps(c, std::integral_constant<int, 1>{});
        c += 16;
    }
    if (c < d) {
        const f16x8 q = *reinterpret_cast<const f16x8*>(qrow + c + kb);
#pragma unroll
        for (int u = 0; u < U; ++u) mul(q, load_k(row[u], c + kb, d), acc[u]);
    }
}

// The query rows gathered, 8 channels per thread, where they are too long for the statistics kernel to do it.
__global__ __launch_bounds__(kThreads) void kvstar_pack_kernel(KvArgs a)
{
    const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    const int per_row = a.dp / 8;
    const int64_t row = i / per_row;
    if (row >= (int64_t)a.items * 32) return;
    const int c = (int)(i - row * per_row) * 8;
    *reinterpret_cast<f16x8*>(a.qp + row * a.dp + c) = load_q(q_row(a, (int)(row >> 5), (int)(row & 31)), c, a.d, a.d_orig);
}

// The query rows of a workgroup's two items into LDS, eight threads per row, each taking every eighth channel, in two
// parts: the channels' numbers are asked for in front of the keys, so that waiting for them is not waiting for those.
template <int KS>
struct Gather {
    QRow q;
    int rl;
    int64_t src[2 * KS];
    __device__ __forceinline__ explicit Gather(const KvArgs& a)
    {
        rl = threadIdx.x >> 3;  // 0 .. 63: row rl % 32 of the workgroup's item rl / 32
        q = q_row(a, blockIdx.y * stat_items(KS) + (rl >> 5), rl & 31);
#pragma unroll
        for (int i = 0; i < 2 * KS; ++i) {
            const int j = (threadIdx.x & 7) + 8 * i;
            src[i] = q.pruned ? q.pruned[j] : j;
        }
    }
    __device__ __forceinline__ void rows(const KvArgs& a, _Float16* qt, int pitch) const
    {
        _Float16 v[2 * KS];
#pragma unroll
        for (int i = 0; i < 2 * KS; ++i) v[i] = q.row[src[i] < 0 ? 0 : (src[i] >= a.d_orig ? a.d_orig - 1 : src[i])];
#pragma unroll
        for (int i = 0; i < 2 * KS; ++i) qt[rl * pitch + (threadIdx.x & 7) + 8 * i] = q.ok ? v[i] : (_Float16)0;
    }
};

// grid = (chunks, ceil(items / kItems)).  Wave w serves row tile w % kItems and every
// kSubs-th tile of representatives of the chunk.  Representatives are the A operand (lane:
// representative lane % 32, channels 8 (lane / 32) .. + 7 of the k-step), query rows the B operand:
// accumulator v of a lane is the score of row lane % 32 against representative
// 8 (v / 4) + 4 (lane / 32) + v % 4 of the tile, so a row's statistics are one lane's work and meet
// once, at the end.  KS = d / 16 for 32, 64 and 128 channels: the loads of several tiles go out
// together, in front of the gather of the query rows (which all waves share through LDS).  Any other d: one
// row tile per workgroup, as many k-steps as the registers take at a time.  Query rows gathered by every lane in
// front of every tile cost 2 to 6 times the call: 8 x 32 query rows, 253 blocks of 64, 96 channels 66 us, gathered
// once 27 us; blocks of 16, 512 channels 208 and 35 us.
template <int KS>
__global__ __launch_bounds__(kThreads) void kvstar_stats_kernel(KvArgs a)
{
    constexpr int kItems = stat_items(KS), kSubs = kThreads / 64 / kItems;  // kSubs waves share a row tile's representatives
    constexpr int U = KS == 2 || KS == 4 ? 2 : 1;  // tiles in flight per wave
    extern __shared__ __align__(16) _Float16 qt[];  // [kItems * 32][pitch], but for kPacked
    const int pitch = (KS > 0 ? KS * 16 : a.dp) + 8;  // 16 bytes of padding spread the rows over the banks
    __shared__ Stat red[kThreads / 64][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = wave % kItems, sub = wave / kItems;
    const int item = blockIdx.y * kItems + li;
    const int h = item < a.items ? item / a.tiles_q : 0;
    const int kb = (lane >> 5) * 8;
    const int t0 = blockIdx.x * a.per_chunk + sub;
    int t1 = (blockIdx.x + 1) * a.per_chunk;
    t1 = item < a.items ? (t1 < a.tiles_k ? t1 : a.tiles_k) : 0;
    auto k_row = [&](int t) {
        int64_t s = (int64_t)t * 32 + (lane & 31);
        s = s < a.S ? s : a.S - 1;
        return a.k + (s * a.Hkv + h) * a.d;
    };
    f16x8 early[kEarly];  // of the first tile, requested in front of the gather
    const bool hurry = a.d <= kEarlyMost;
    f16x8 kk[U][KS > 0 ? KS : 1];
    auto load_tiles = [&](int t) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const _Float16* row = k_row(t + u * kSubs < t1 ? t + u * kSubs : t);
#pragma unroll
            for (int c = 0; c < KS; ++c) kk[u][c] = *reinterpret_cast<const f16x8*>(row + c * 16 + kb);
        }
    };
    if constexpr (KS > 0) {
        const Gather<KS> gather(a);
        load_tiles(t0 < a.tiles_k ? t0 : 0);
        gather.rows(a, qt, pitch);
    } else if constexpr (KS == kAnyDim) {
        const _Float16* row = k_row(t0 < a.tiles_k ? t0 : 0);
#pragma unroll
        for (int i = 0; i < kEarly; ++i) {
            early[i] = f16x8{0};
            if (hurry && 16 * i + 16 <= a.d) early[i] = *reinterpret_cast<const f16x8u*>(row + 16 * i + kb);
        }
        // sixteen threads per query row, each taking every sixteenth channel
        const int rl = threadIdx.x >> 4;
        const QRow q = q_row(a, blockIdx.y, rl);
        for (int c = threadIdx.x & 15; c < a.dp; c += 16 * 8) {
            int64_t src[8];
            _Float16 v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) src[i] = q_channel(q, c + 16 * i < a.d ? c + 16 * i : 0, a.d_orig);
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = q.row[src[i]];
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (c + 16 * i < a.dp) qt[rl * pitch + c + 16 * i] = q.ok && c + 16 * i < a.d ? v[i] : (_Float16)0;
        }
    }
    if constexpr (KS != kPacked) {
        __syncthreads();
        if (blockIdx.x == 0) {  // the gathered rows, for the mass kernel
            const int per_row = KS > 0 ? 2 * KS : a.dp / 8;
            for (int i = threadIdx.x; i < kItems * 32 * per_row; i += kThreads) {
                const int r = i / per_row, c = (i % per_row) * 8;
                const int64_t row = (int64_t)blockIdx.y * kItems * 32 + r;
                if (row < (int64_t)a.items * 32)
                    *reinterpret_cast<f16x8*>(a.qp + row * a.dp + c) = *reinterpret_cast<const f16x8*>(qt + r * pitch + c);
            }
        }
    }
    float m = -INFINITY, sum = 0.0f;
    // the scores of U tiles (t, t + kSubs, ...) join the row's statistics
    auto add_tiles = [&](const f32x16 (&acc)[U], int t) {
        float x[U][16];
        float nm = m;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t s0 = (int64_t)(t + u * kSubs) * 32;
            const bool whole = t + u * kSubs < t1 && s0 + 32 <= a.S;  // uniform
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                x[u][v] = acc[u][v];
                if (!whole && (t + u * kSubs >= t1 || s0 + 8 * (v / 4) + 4 * (lane >> 5) + v % 4 >= a.S))
                    x[u][v] = -INFINITY;
                nm = fmaxf(nm, x[u][v]);
            }
        }
        // a lane that has seen no number yet measures from 0: minus infinities add 0, a NaN (which the
        // maximum passes over) still makes the row's sum one
        const float base = stat_base(nm);
        float cs = 0.0f;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int v = 0; v < 16; ++v) cs += exp_small(x[u][v] - base);
        sum = sum * exp_small(m - base) + cs;
        m = nm;
    };
    for (int t = t0; t < t1; t += U * kSubs) {
        f32x16 acc[U];
#pragma unroll
        for (int u = 0; u < U; ++u) acc[u] = f32x16{0};
        if constexpr (KS > 0) {
            if (t != t0) load_tiles(t);
            const _Float16* qrow = qt + (li * 32 + (lane & 31)) * pitch + kb;
#pragma unroll
            for (int c = 0; c < KS; ++c) {
                const f16x8 qq = *reinterpret_cast<const f16x8*>(qrow + c * 16);
#pragma unroll
                for (int u = 0; u < U; ++u) acc[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kk[u][c], qq, acc[u], 0, 0, 0);
            }
        } else {
            const _Float16* row[U];
#pragma unroll
            for (int u = 0; u < U; ++u) row[u] = k_row(t + u * kSubs < t1 ? t + u * kSubs : t);
            if constexpr (KS == kPacked) {
                dots_any<false>(a.qp + ((int64_t)item * 32 + (lane & 31)) * a.dp, row, kb, 0, a.d, acc);
            } else {
                const _Float16* qrow = qt + (lane & 31) * pitch;
                int c = 0;
                if (hurry && t == t0) {
#pragma unroll
                    for (int i = 0; i < kEarly; ++i) {
                        if (16 * i + 16 > a.d) break;
                        acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(early[i], *reinterpret_cast<const f16x8*>(qrow + 16 * i + kb), acc[0], 0, 0, 0);
                        c = 16 * i + 16;
                    }
                }
                dots_any<false>(qrow, row, kb, c, a.d, acc);
            }
        }
        add_tiles(acc, t);
    }
    red[wave][lane] = Stat{m, sum};  // a row is lanes r and r + 32 of kSubs waves
    __syncthreads();
    if (sub == 0 && lane < 32 && item < a.items) {
        Stat v[2 * kSubs];
#pragma unroll
        for (int i = 0; i < 2 * kSubs; ++i) v[i] = red[li + i / 2 * kItems][lane + 32 * (i & 1)];
        a.part[(int64_t)blockIdx.x * a.items * 32 + item * 32 + lane] = merge(Stat{-INFINITY, 0.0f}, v);
    }
}

// One workgroup per group of blocks (a block of 32 and more representatives, or as many small blocks as
// 32 representatives make): the rows' statistics merged from the chunks' pairs, then each wave takes
// every eighth row tile against the group's representatives, now as the B operand: accumulator v of a
// lane is row 8 (v / 4) + 4 (lane / 32) + v % 4 against representative lane % 32, whose probabilities
// add up in the lane.  Partial sums meet in a fixed order: accumulators, row tiles of a wave, lane
// halves, waves, representatives.
template <int KS, bool EARLY>
__global__ __launch_bounds__(kThreads) void kvstar_mass_kernel(KvArgs a)
{
    constexpr int kWaves = kThreads / 64;
    __shared__ __align__(16) float2 stat[kMassRows];  // (largest score, 1 / sum of exponentials) of a row
    __shared__ Stat halves[kThreads];
    __shared__ float red[kWaves][32];
    __shared__ float rep[32];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int kb = (lane >> 5) * 8;
    const int rows = a.items * 32;
    const int batches = (rows + kMassRows - 1) / kMassRows;
    const int real = a.X * a.g;  // query rows of a KV head
    for (int grp = blockIdx.x; grp < a.groups; grp += gridDim.x) {
        const int64_t s0 = (int64_t)grp * a.group_blocks * a.M;  // the group's first representative
        const int64_t left = a.S - s0;
        const int64_t want = (int64_t)a.group_blocks * a.M;
        const int ns = (int)(left < want ? left : want);
        float tot = 0.0f;
        auto rep_row = [&](int t, int h) {  // representative lane % 32 of tile t of the group
            const int s = t * 32 + (lane & 31);
            return a.k + ((s0 + (s < ns ? s : ns - 1)) * a.Hkv + h) * a.d;
        };
        f16x8 early[2][EARLY ? kEarly : 1];  // of the first two tiles, requested in front of the statistics
        if constexpr (EARLY) {
            const int h = wave < a.items ? wave / a.tiles_q : 0;
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int i = 0; i < kEarly; ++i) early[u][i] = *reinterpret_cast<const f16x8u*>(rep_row(u, h) + 16 * i + kb);
        }
        for (int batch = 0; batch < batches; ++batch) {
            const int r0 = batch * kMassRows;
            const int nr = rows - r0 < kMassRows ? rows - r0 : kMassRows;
            if (batches > 1 || grp == (int)blockIdx.x) {
                // two threads per row where the rows leave half of the workgroup idle
                const bool split = nr <= kThreads / 2;
                const int step = split ? kThreads / 2 : kThreads;
                const int half = split ? __builtin_amdgcn_readfirstlane(threadIdx.x / (kThreads / 2)) : 0;
                const int c_mid = split ? (a.chunks + 1) / 2 : a.chunks;
                const int c0 = half ? c_mid : 0, c1 = half ? a.chunks : c_mid;
                for (int r = split ? threadIdx.x % (kThreads / 2) : threadIdx.x; r < (split ? step : nr); r += step) {
                    Stat st{-INFINITY, 0.0f};
                    if (r < nr) {
                        const Stat* p = a.part + r0 + r;
                        int c = c0;
                        for (; c + 16 <= c1; c += 16) {
                            Stat v[16];
#pragma unroll
                            for (int i = 0; i < 16; ++i) v[i] = p[(int64_t)(c + i) * rows];
                            st = merge(st, v);
                        }
                        for (; c < c1; c += 8) {
                            Stat v[8];
#pragma unroll
                            for (int i = 0; i < 8; ++i) v[i] = p[(int64_t)(c + i < c1 ? c + i : c1 - 1) * rows];
                            st = merge(st, v, c1 - c);
                        }
                    }
                    if (split) {
                        halves[threadIdx.x] = st;
                        __syncthreads();
                        if (half == 0) {
                            const Stat other[1] = {halves[threadIdx.x + kThreads / 2]};
                            st = merge(st, other);
                        }
                    }
                    // the reference normalises only when the sum exceeds 1e-9
                    if (half == 0 && r < nr) stat[r] = make_float2(st.m, st.s > 1e-9f ? 1.0f / st.s : 1.0f);
                }
                __syncthreads();
            }
            const int items = nr / 32;
            for (int it = wave; it < items; it += kWaves) {
                const int item = r0 / 32 + it;
                const int h = item / a.tiles_q;
                const int valid = real - (item - h * a.tiles_q) * 32;  // rows of the tile that exist
                const _Float16* qrow = a.qp + ((int64_t)item * 32 + (lane & 31)) * (KS > 0 ? KS * 16 : a.dp);
                f16x8 qq[KS > 0 ? KS : 1];
#pragma unroll
                for (int c = 0; c < KS; ++c) qq[c] = *reinterpret_cast<const f16x8*>(qrow + c * 16 + kb);
                auto add_tile = [&](const f32x16& acc, int t) {
                    float p = 0.0f;
#pragma unroll
                    for (int v4 = 0; v4 < 4; ++v4) {
                        const int row = 8 * v4 + 4 * (lane >> 5);
                        const float4 sa = *reinterpret_cast<const float4*>(&stat[it * 32 + row]);
                        const float4 sb = *reinterpret_cast<const float4*>(&stat[it * 32 + row + 2]);
                        const float mm[4] = {sa.x, sa.z, sb.x, sb.z}, inv[4] = {sa.y, sa.w, sb.y, sb.w};
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float e = exp_small(acc[v4 * 4 + i] - mm[i]) * inv[i];
                            p += valid >= 32 || row + i < valid ? e : 0.0f;
                        }
                    }
                    if (t * 32 + (lane & 31) < ns) tot += p;
                };
                for (int t = 0; t * 32 < ns; t += 2) {
                    if constexpr (KS > 0) {
                        f16x8 kk[2][KS];
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            const _Float16* row = rep_row(t + u, h);
#pragma unroll
                            for (int c = 0; c < KS; ++c) kk[u][c] = *reinterpret_cast<const f16x8*>(row + c * 16 + kb);
                        }
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            if ((t + u) * 32 >= ns) break;
                            f32x16 acc = {0};
#pragma unroll
                            for (int c = 0; c < KS; ++c)
                                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(qq[c], kk[u][c], acc, 0, 0, 0);
                            add_tile(acc, t + u);
                        }
                    } else {
                        auto tiles = [&](auto n_) {
                            constexpr int U = decltype(n_)::value;
                            const _Float16* row[U];
                            f32x16 acc[U];
#pragma unroll
                            for (int u = 0; u < U; ++u) {
                                row[u] = rep_row(t + u, h);
                                acc[u] = f32x16{0};
                            }
                            int c = 0;
                            if constexpr (EARLY) {
                                if (t == 0 && item == wave) {
                                    f16x8 q[kEarly];
#pragma unroll
                                    for (int i = 0; i < kEarly; ++i) q[i] = *reinterpret_cast<const f16x8*>(qrow + 16 * i + kb);
#pragma unroll
                                    for (int i = 0; i < kEarly; ++i)
#pragma unroll
                                        for (int u = 0; u < U; ++u)
                                            acc[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(q[i], early[u][i], acc[u], 0, 0, 0);
                                    c = 16 * kEarly;
                                }
                            }
                            dots_any<true>(qrow, row, kb, c, a.d, acc);
#pragma unroll
                            for (int u = 0; u < U; ++u) add_tile(acc[u], t + u);
                        };
                        if ((t + 1) * 32 < ns) tiles(std::integral_constant<int, 2>{});
                        else tiles(std::integral_constant<int, 1>{});
                    }
                }
            }
            if (batches > 1) __syncthreads();  // the next batch overwrites the statistics
        }
        tot += __shfl_xor(tot, 32);
        if (lane < 32) red[wave][lane] = tot;
        __syncthreads();
        if (wave == 0) {
            float t = 0.0f;
            if (lane < 32) {
#pragma unroll
                for (int w = 0; w < kWaves; ++w) t += red[w][lane];
                rep[lane] = t;
            }
            __builtin_amdgcn_wave_barrier();
            if (a.M >= 32) {
                // every lane's representatives belong to the one block
#pragma unroll
                for (int o = 16; o >= 1; o >>= 1) t += __shfl_xor(t, o);
                if (lane == 0) a.keys[grp] = score_key(t);
            } else {
                const int blk = grp * a.group_blocks + lane;
                if (lane < a.group_blocks && blk < a.n_blocks) {
                    float s = 0.0f;
                    for (int i = 0; i < a.M; ++i) s += rep[lane * a.M + i];
                    a.keys[blk] = score_key(s);
                }
            }
        }
        __syncthreads();
    }
}

// Blocks whose q.k is taken once.  This kernel leaves the maximum and the sum of exponentials of every (row, block), and kvstar_merge_kernel, which
// sees all of a row's blocks, makes probabilities of them.
// grid = (parts of the blocks, ceil(items / 2)).  Operands as in kvstar_stats_kernel.  A wave takes a block, or as many
// small ones as two tiles hold (one tile of 128 channels: registers), at a time.
template <int KS, int UNIT>
__global__ __launch_bounds__(kThreads) void kvstar_unit_kernel(ucm::ArgPair qk, ucm::ArgPair early, ucm::ArgInts n, int X, KvArgs a)
{
    a.q = ucm::arg_ptr<const _Float16>(qk.x); a.k = ucm::arg_ptr<const _Float16>(qk.y); a.pruned = ucm::arg_ptr<const int64_t>(early.x);
    a.S = ucm::arg_lo(early.y); a.Hkv = ucm::arg_hi(early.y); a.Hq = n.x & 0xffff; a.g = (int)((uint32_t)n.x >> 16); a.d_orig = n.y;
    a.tiles_q = n.z; a.items = n.w; a.X = X; a.d = KS * 16; a.tiles_k = (int)(a.S + 31) / 32;
    constexpr int kItems = stat_items(KS), kSubs = kThreads / 64 / kItems;
    constexpr int U = UNIT == 64 || KS <= 4 ? 2 : 1;
    constexpr int pitch = KS * 16 + 8;
    __shared__ __align__(16) _Float16 qt[kItems * 32 * pitch];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = wave % kItems, sub = wave / kItems;
    const int item = blockIdx.y * kItems + li;
    const int h = item < a.items ? (a.tiles_q == 1 ? item : item / a.tiles_q) : 0;
    const int kb = (lane >> 5) * 8;
    const int rows = a.items * 32;
    const int per = UNIT == 64 ? a.M / 64 : 1;  // steps of two tiles to a block
    const int steps = item < a.items ? (UNIT == 64 ? a.units : (a.tiles_k + U - 1) / U) : 0;
    const int p0 = blockIdx.x * kSubs + sub;
    f16x8 kk[U][KS];
    auto load_tiles = [&](int p) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int64_t s = (int64_t)(p * U + u) * 32 + (lane & 31);
            s = s < a.S ? s : a.S - 1;
            const _Float16* row = a.k + (s * a.Hkv + h) * (KS * 16);
#pragma unroll
            for (int c = 0; c < KS; ++c) kk[u][c] = *reinterpret_cast<const f16x8*>(row + c * 16 + kb);
        }
    };
    const Gather<KS> gather(a);
    load_tiles(p0 < steps ? p0 * per : 0);
    gather.rows(a, qt, pitch);
    __syncthreads();
    Stat* out = a.part + item * 32 + (lane & 31);
    Stat sofar{-INFINITY, 0.0f};
    for (int p = p0, q = 0; p < steps; q + 1 < per ? ++q : (p += gridDim.x * kSubs, q = 0)) {
        if (p != p0 || q != 0) load_tiles(p * per + q);
        f32x16 acc[U];
#pragma unroll
        for (int u = 0; u < U; ++u) acc[u] = f32x16{0};
        const _Float16* qrow = qt + (li * 32 + (lane & 31)) * pitch + kb;
#pragma unroll
        for (int c = 0; c < KS; ++c) {
            const f16x8 qq = *reinterpret_cast<const f16x8*>(qrow + c * 16);
#pragma unroll
            for (int u = 0; u < U; ++u) acc[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kk[u][c], qq, acc[u], 0, 0, 0);
        }
        // a unit's tile values lo .. hi - 1 of both lane halves; a unit is whole (S is a whole number of them)
        auto pair_of = [&](auto get, int n) {
            float m = -INFINITY;
#pragma unroll
            for (int v = 0; v < n; ++v) m = fmaxf(m, get(v));
            m = fmaxf(m, __shfl_xor(m, 32));
            // minus infinities alone measure from 0 and add 0; a NaN, which the maximum passes over, makes the sum one
            const float base = stat_base(m);
            ucm::ExpSum sum;
#pragma unroll
            for (int v = 0; v < n; ++v)
                sum.add(__builtin_elementwise_maximum(get(v) - base, -200.0f), [](float t) { return __builtin_amdgcn_exp2f(t); });
            const float s = sum.sum();
            return Stat{m, s + __shfl_xor(s, 32)};
        };
        if constexpr (UNIT == 64) {
            const Stat st = pair_of([&](int v) { return acc[v / 16][v % 16]; }, 32);
            sofar = q == 0 ? st : join(sofar, st);
            if (lane < 32 && q == per - 1) out[(int64_t)p * rows] = sofar;
        } else {
            constexpr int N = UNIT / 2, kPer = 32 / UNIT;
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < kPer; ++i) {
                    const int unit = (p * U + u) * kPer + i;
                    const Stat st = pair_of([&](int v) { return acc[u][i * N + v]; }, N);
                    if (lane < 32 && unit < a.units) out[(int64_t)unit * rows] = st;
                }
        }
    }
}

// The other half: grid = items * 32 / kMergeRows, a workgroup per kMergeRows query rows of an item.  A thread holds
// R units of one row at a time: the row's maximum and sum over all units meet through the lanes and LDS, then every
// unit's probability is its sum times exp(its maximum - the row's) over the row's sum, added up over the rows by the
// sixteen lanes that hold them.
template <int NT, int R>
__global__ __launch_bounds__(NT) void kvstar_merge_kernel(ucm::ArgPair in_out, ucm::ArgInts n)
{
    const Stat* const part = ucm::arg_ptr<const Stat>(in_out.x);
    float* const sums = ucm::arg_ptr<float>(in_out.y);
    const int units = n.x, items = n.y, tiles_q = n.z, real_rows = n.w;
    constexpr int kGroups = NT / kMergeRows, kWaves = NT / 64;
    static_assert(kMergeRows == 16 && kWaves % 4 == 0, "a row of lanes");
    __shared__ Stat red[kWaves][kMergeRows];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = threadIdx.x % kMergeRows, grp = threadIdx.x / kMergeRows;
    const int rows = items * 32, r0 = blockIdx.x * kMergeRows;
    const int item = r0 / 32;
    // rows of the item that exist: X * g of the KV head are cut into its tiles
    const bool real = (item % tiles_q) * 32 + r0 % 32 + r < real_rows;
    const Stat* p = part + r0 + r;
    Stat v[R];
    auto load = [&](int u0) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int u = u0 + grp + i * kGroups;
            v[i] = p[(int64_t)(u < units ? u : units - 1) * rows];
        }
#pragma unroll
        for (int i = 0; i < R; ++i)
            if (u0 + grp + i * kGroups >= units) v[i] = Stat{-INFINITY, 0.0f};
    };
    Stat st{-INFINITY, 0.0f};
    // one load: v[i].s becomes the unit's sum measured from the thread's own largest score
    const bool held = units <= R * kGroups;
    if (held) {
        load(0);
#pragma unroll
        for (int i = 0; i < R; ++i) st.m = fmaxf(st.m, v[i].m);
        const float base = stat_base(st.m);
#pragma unroll
        for (int i = 0; i < R; ++i) {
            v[i].s *= exp_small(v[i].m - base);
            st.s += v[i].s;
        }
    } else {
        for (int u0 = 0; u0 < units; u0 += R * kGroups) {
            load(u0);
            st = merge(st, v);
        }
    }
    const float own = st.m;
    auto meet = [&] {  // the four threads of a wave that share a row
#pragma unroll
        for (int o = kMergeRows; o < 64; o <<= 1) {
            const Stat other[1] = {Stat{__shfl_xor(st.m, o), __shfl_xor(st.s, o)}};
            st = merge(st, other);
        }
    };
    meet();
    if (lane < kMergeRows) red[wave][lane] = st;
    __syncthreads();
    // every thread a quarter of the waves: exponentials are what this kernel issues most of
    Stat all[kWaves / 4];
#pragma unroll
    for (int w = 0; w < kWaves / 4; ++w) all[w] = red[lane / kMergeRows * (kWaves / 4) + w][r];
    st = merge(Stat{-INFINITY, 0.0f}, all);
    meet();
    // the reference normalises only when the sum exceeds 1e-9
    float inv = st.s > 1e-9f ? 1.0f / st.s : 1.0f;
    if (st.m == -INFINITY) inv = NAN;  // a row of minus infinities has no probabilities
    const float scale = own == st.m ? 1.0f : exp_small(own - st.m);
    for (int u0 = 0; u0 < units; u0 += R * kGroups) {
        if (!held) load(u0);
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int u = u0 + grp + i * kGroups;
            float e = real ? v[i].s * (held ? scale : exp_small(v[i].m - st.m)) * inv : 0.0f;
            auto add = [&](auto ctl) {
                e += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(e), decltype(ctl)::value, 0xf, 0xf, false));
            };
            add(std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
            add(std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
            add(std::integral_constant<int, 0x141>{});  // row_half_mirror
            add(std::integral_constant<int, 0x140>{});  // row_mirror
            if (r == 0 && u < units) sums[(int64_t)blockIdx.x * units + u] = e;
        }
    }
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

constexpr int kMaxDim = 1024;

// How the representatives are shared out: the larger d, the more chunks.
void plan_chunks(KvArgs& a)
{
    a.S = (int64_t)a.n_blocks * a.M;
    a.tiles_k = (int)ucm::ceil_div(a.S, 32);
    // kMaxChunks: 32 leave half of the chip idle at 8 KV heads (statistics 8.9 us instead of 7.2), and every
    // workgroup of the mass kernel reads all chunks' pairs of its rows.  Fewer than eight tiles to a workgroup
    // of the statistics kernel, and fewer than 32 representatives to one of the mass kernel, only make more
    // pairs to merge (1000 blocks of one representative, 32 channels: 15.0 us, in 256 groups 16.3) unless rows
    // are long and compute units idle (512 channels, 253 blocks of 16: 40.6 us, like this 34.9; 256 channels,
    // 64 blocks of 16, two heads: 19.2 and 17.0).
    const bool longer = a.d > kLongDim;
    a.per_chunk = (int)ucm::ceil_div(a.tiles_k, kMaxChunks);
    if (a.per_chunk < (longer ? kLeastTiles : 8)) a.per_chunk = longer ? kLeastTiles : 8;
    a.chunks = (int)ucm::ceil_div(a.tiles_k, a.per_chunk);
    a.group_blocks = a.M >= 32 ? 1 : 32 / a.M;
    if (longer)
        while (a.group_blocks > 1 && ucm::ceil_div(a.n_blocks, a.group_blocks) < 256) a.group_blocks /= 2;
    a.groups = (int)ucm::ceil_div(a.n_blocks, a.group_blocks);
}

// Query rows with their padding, for every number of KV heads: at most 31 rows of it to each.
int64_t padded_rows(const KvArgs& a) { return (int64_t)a.Hq * (a.X + 31); }

// Whether the blocks are units: whole halves, ones or pairs of tiles, so that a wave has all of a block's scores.
// A pair is 8 bytes for every row, written and read, where the second way reads a block's keys and takes its products
// again: at 16 representatives of 32 channels that is even (256 rows, 1024 blocks 20.5 and 21.4 us, 2040: 27.7 and
// 27.5), at 64 it never is (2000: 39.3 and 53.8).  Blocks of 48 in units of 16: 20.5 and 18.0.
void plan_units(KvArgs& a)
{
    const bool whole = a.M == 16 || a.M == 32 || (a.M % 64 == 0 && a.M <= 256);
    const int most = a.M == 16 ? 1024 : kRankSums;
    a.units = whole && a.n_blocks <= most && a.n_blocks * padded_rows(a) * 8 <= kUnitBytes ? a.n_blocks : 0;
}

// Addresses of the workspace's parts, of the second way with `chunks` chunks and of the units for `rows` rows.
size_t carve_kvstar(KvArgs& a, void* base, int chunks)
{
    const size_t rows = (size_t)padded_rows(a);
    char* p = (char*)base;
    size_t off = 0;
    a.qp = (_Float16*)(p + off);
    off += align256(rows * kMaxDim * 2);
    a.part = (Stat*)(p + off);
    off += align256((size_t)chunks * rows * 8);
    a.keys = (uint32_t*)(p + off);
    off += align256((size_t)key_pitch(a.n_blocks) * 4);
    return off;
}

size_t carve_units(KvArgs& a, void* base, int64_t rows)
{
    char* p = (char*)base;
    a.part = (Stat*)p;
    const size_t off = align256((size_t)a.units * rows * 8);
    a.sums = (float*)(p + off);
    return off + align256(ucm::ceil_div(rows, kMergeRows) * (size_t)a.units * 4);
}

template <int KS>
int launch_kvstar(const KvArgs& a, hipStream_t st)
{
    int rc;
    if (KS == kPacked) {
        hipLaunchKernelGGL(kvstar_pack_kernel, dim3((unsigned)ucm::ceil_div((int64_t)a.items * 4 * a.dp, kThreads)), dim3(kThreads), 0, st, a);
        rc = ucm::launch_status("kvstar_pack_kernel");
        if (rc != UCM_OK) return rc;
    }
    const size_t lds = KS == kPacked ? 0 : (size_t)stat_items(KS) * 32 * (a.dp + 8) * 2;
    hipLaunchKernelGGL(kvstar_stats_kernel<KS>, dim3((unsigned)a.chunks, (unsigned)ucm::ceil_div(a.items, stat_items(KS))),
                       dim3(kThreads), lds, st, a);
    rc = ucm::launch_status("kvstar_stats_kernel");
    if (rc != UCM_OK) return rc;
    const dim3 groups((unsigned)(a.groups < kMassGroups ? a.groups : kMassGroups));
    // Early loads where a block has two tiles and long rows and one generation of workgroups has nothing else to
    // hide them behind (253 blocks of 64, 192 channels: 38.1 and 36.3 us); elsewhere their registers cost more
    // (1024 blocks of 32, 96 channels: 59.5 and 69.4 us).
    if (KS == kAnyDim && a.M > 32 && a.d >= 16 * kEarly && a.groups <= 256)
        hipLaunchKernelGGL((kvstar_mass_kernel<kAnyDim, true>), groups, dim3(kThreads), 0, st, a);
    else
        hipLaunchKernelGGL((kvstar_mass_kernel<(KS > 0 ? KS : kAnyDim), false>), groups, dim3(kThreads), 0, st, a);
    return ucm::launch_status("kvstar_mass_kernel");
}

template <int KS, int UNIT>
int launch_units(const KvArgs& a, hipStream_t st)
{
    constexpr int U = UNIT == 64 || KS <= 4 ? 2 : 1, kSubs = kThreads / 64 / stat_items(KS);
    const int64_t heads = ucm::ceil_div(a.items, stat_items(KS)), most = kUnitGroups / heads;
    const int64_t need = ucm::ceil_div(UNIT == 64 ? a.units : ucm::ceil_div(a.tiles_k, U), kSubs);
    const int64_t parts = need < most ? need : (most < 1 ? 1 : most);
    hipLaunchKernelGGL((kvstar_unit_kernel<KS, UNIT>), dim3((unsigned)parts, (unsigned)heads), dim3(kThreads), 0, st,
                       ucm::arg_pair(a.q, a.k), ucm::arg_pair(a.pruned, ucm::arg_words((int)a.S, a.Hkv)),
                       ucm::ArgInts{(int)((uint32_t)a.Hq | (uint32_t)a.g << 16), a.d_orig, a.tiles_q, a.items}, a.X, a);  // X * Hq <= 65535
    int rc = ucm::launch_status("kvstar_unit_kernel");
    if (rc != UCM_OK) return rc;
    const dim3 grid((unsigned)(a.items * (32 / kMergeRows)));
    auto launch = [&](auto kernel, int threads) {
        hipLaunchKernelGGL(kernel, grid, dim3((unsigned)threads), 0, st, ucm::arg_pair(a.part, a.sums),
                           ucm::ArgInts{a.units, a.items, a.tiles_q, a.X * a.g});
    };
    if (a.units <= 256) launch(kvstar_merge_kernel<512, 8>, 512);
    else if (a.units <= 512) launch(kvstar_merge_kernel<1024, 8>, 1024);
    else launch(kvstar_merge_kernel<1024, 16>, 1024);
    return ucm::launch_status("kvstar_merge_kernel");
}

template <int KS>
int launch_units(const KvArgs& a, hipStream_t st)
{
    return a.M == 16 ? launch_units<KS, 16>(a, st) : a.M == 32 ? launch_units<KS, 32>(a, st) : launch_units<KS, 64>(a, st);
}

}  // namespace

extern "C" size_t ucm_kvstar_topk_workspace_bytes(int32_t X, int32_t Hq, int64_t n_blocks, int32_t M)
{
    if (X <= 0 || Hq <= 0 || n_blocks <= 0 || M <= 0) return 256;
    if (n_blocks > INT32_MAX || n_blocks * M > INT32_MAX) return 256;  // refused by the call
    KvArgs a{};
    a.X = X; a.Hq = Hq; a.n_blocks = (int)n_blocks; a.M = M;
    plan_units(a);
    // the most chunks that any dimension has for as many representatives or fewer
    const int64_t chunks = ucm::ceil_div(ucm::ceil_div(n_blocks * M, 32), kLeastTiles);
    const size_t general = carve_kvstar(a, nullptr, (int)(chunks < kMaxChunks ? chunks : kMaxChunks)), units = carve_units(a, nullptr, padded_rows(a));
    return general > units ? general : units;
}

extern "C" int ucm_kvstar_topk(const void* query, int32_t X, int32_t Hq, int32_t d_orig,
                               const void* blk_repre, int64_t n_blocks, int32_t M, int32_t Hkv,
                               int32_t d, const int64_t* pruned_index, int32_t topk,
                               int32_t* out_idx, float* out_score, void* workspace,
                               size_t workspace_bytes, ucm_stream_t stream)
{
    ucm::clear_error();
    UCM_REQUIRE(query && blk_repre && out_idx && out_score, "null pointer");
    UCM_REQUIRE(X > 0 && Hq > 0 && Hkv > 0 && d > 0 && d_orig > 0 && n_blocks > 0 && M > 0,
                "non-positive shape");
    UCM_REQUIRE(Hq % Hkv == 0, "Num_q_heads must be a divisible by num_kv_heads.");
    UCM_REQUIRE(pruned_index || d == d_orig,
                "Dimension mismatch: No dPrunedIndex, but Q and K head dims differ.");
    UCM_REQUIRE(topk > 0, "topk %d must be positive", topk);
    if (topk > kMaxTopk) return ucm::fail(UCM_EUNSUPPORTED, "topk %d above %d", topk, kMaxTopk);
    UCM_REQUIRE(d <= kMaxDim, "head dim %d above %d", d, kMaxDim);
    UCM_REQUIRE(n_blocks <= INT32_MAX && n_blocks * M <= INT32_MAX, "too many block representatives");
    const int64_t rows = (int64_t)X * Hq;
    // row tiles are a grid dimension; the second bound is the entry point's own, no index comes near it
    UCM_REQUIRE(rows <= 65535 && rows * M <= INT32_MAX, "too many query rows");
    UCM_REQUIRE((((uintptr_t)blk_repre | (uintptr_t)workspace) & 15) == 0, "block representatives must be 16-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    KvArgs a{};
    a.q = (const _Float16*)query; a.k = (const _Float16*)blk_repre; a.pruned = pruned_index;
    a.X = X; a.Hq = Hq; a.Hkv = Hkv; a.g = Hq / Hkv; a.d_orig = d_orig; a.d = d; a.dp = (int)ucm::ceil_div(d, 16) * 16;
    a.n_blocks = (int)n_blocks; a.M = M;
    a.tiles_q = (int)ucm::ceil_div((int64_t)X * a.g, 32);
    a.items = Hkv * a.tiles_q;
    plan_units(a);
    a.d = kMaxDim;  // as much for every dimension
    plan_chunks(a);
    UCM_REQUIRE(workspace && workspace_bytes >= carve_kvstar(a, nullptr, a.chunks), "workspace too small");
    a.d = d;
    plan_chunks(a);
    SortArgs s{};
    s.max_n = (int)n_blocks; s.topk = topk;
    s.out_idx = out_idx; s.out_score = out_score;
    // Few row tiles leave the merging to few workgroups.  Four tiles, 600 blocks of 16 x 32 channels: 18.6 and the second way 17.0 us;
    // larger blocks have more to gain: one tile, 300 of 16 x 64 channels 15.4 and 17.0, 253 of 32 x 32 13.0 and 14.4, 24 of 32 x 32 12.9
    // and 14.1, 1500 of 32 x 32 23.9 and 24.5; eight tiles, 600 of 16 x 32 16.8 and 19.0.
    const bool few = M == 16 && d == 32 && a.items < 8;
    // (a buffer that only the second way fits into, one asked for at another shape, is taken by it)
    if (a.units > 0 && !few && (d == 32 || d == 64 || d == 128) && carve_units(a, workspace, (int64_t)a.items * 32) <= workspace_bytes) {
        const int rc = d == 32 ? launch_units<2>(a, st) : d == 64 ? launch_units<4>(a, st) : launch_units<8>(a, st);
        if (rc != UCM_OK) return rc;
        return launch_rank_sums(s, a.sums, a.items * (32 / kMergeRows), st);
    }
    carve_kvstar(a, workspace, a.chunks);
    const int rc = d == 32 ? launch_kvstar<2>(a, st)
                 : d == 64 ? launch_kvstar<4>(a, st)
                 : d == 128 ? launch_kvstar<8>(a, st)
                                   : d <= kAnyDimMost ? launch_kvstar<kAnyDim>(a, st)
                                 : launch_kvstar<kPacked>(a, st);
    if (rc != UCM_OK) return rc;
    s.keys = a.keys;
    return launch_topk(s, 1, st);
}
