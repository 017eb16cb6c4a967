// Float retrieval for gfx950: per request, dot products of one query with a list of candidate
// rows of a [n_items, dim] fp32 matrix, then the top-k candidates in descending score order.
//
// GPU counterpart of the reference's ESA retrieval backend
// (ucm/sparse/esa/retrieval/cpy/retrieval_backend.cpp:207-227: for every allowed index a
// sequential fp32 dot product, std::partial_sort by descending score, the first
// min(n_allowed, topk) pairs returned).  Two kernels:
//   * dot_score_kernel — HBM-bound gather: one wave per kRowsPerWave candidate rows, 16-byte loads;
//     writes one order-preserving 32-bit key per candidate (candidates that are -1 or outside the
//     matrix get a key below every number);
//   * launch_topk() (float_topk.h) — one launch selects and orders.  Equal scores come out in list order;
//     the reference leaves ties unspecified.
// Scores differ from the reference's in the last bits (the partial sums are added in a
// different order); the tolerance is stated where the results are compared.
#include <type_traits>

#include "common.h"
#include "float_topk.h"

namespace {

constexpr int kDotThreads = 256;
constexpr int kRowsPerWave = 4;
constexpr int kDotChunks = 4;  // 256-value chunks of a wave's rows requested together

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // a caller's query need not be aligned

struct DotArgs {
    const float* data;
    int64_t n_items;
    int dim;
    const float* q;        // [B][dim]
    const int32_t* idx;    // [B][max_n], -1 = no candidate
    int max_n;
    uint32_t* keys;        // [B] rows, key_pitch(max_n) apart
};

// Sum over the 64 lanes, in lane 63.
__device__ __forceinline__ float wave_sum_last(float v)
{
    auto moved = [](float x, auto ctrl, auto rows) {
        return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), decltype(ctrl)::value,
                                                                     decltype(rows)::value, 0xf, true));
    };
    using std::integral_constant;
    v += moved(v, integral_constant<int, 0xB1>{}, integral_constant<int, 0xf>{});   // quad_perm [1,0,3,2]
    v += moved(v, integral_constant<int, 0x4E>{}, integral_constant<int, 0xf>{});   // quad_perm [2,3,0,1]
    v += moved(v, integral_constant<int, 0x141>{}, integral_constant<int, 0xf>{});  // row_half_mirror
    v += moved(v, integral_constant<int, 0x140>{}, integral_constant<int, 0xf>{});  // row_mirror
    v += moved(v, integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});  // row_bcast:15
    v += moved(v, integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});  // row_bcast:31
    return v;
}

// Bound by HBM: candidates x dim x 4 bytes.  A wave takes four candidate rows and requests up to
// kDotChunks KiB of each before it uses the first (16 loads in flight, 16 KiB per wave; the list entries
// and the query pieces, which come from the caches, go out in front of them), so the row data cost one
// round trip; no LDS and no barrier.  2 x 8000 rows of 1024 (65.5 MB): 12.3 us = 5.3 TB/s of the launch;
// with 4 KiB in flight per wave, behind a barrier for a query staged in LDS, 14.6 us.
__global__ __launch_bounds__(kDotThreads) void dot_score_kernel(ucm::ArgPair rows, ucm::ArgPair lists, ucm::ArgInts n)
{
    const DotArgs a{ucm::arg_ptr<const float>(rows.x), (int64_t)(uint32_t)n.z | (int64_t)n.w << 32, n.x, ucm::arg_ptr<const float>(rows.y),
                    ucm::arg_ptr<const int32_t>(lists.x), n.y, ucm::arg_ptr<uint32_t>(lists.y)};
    const int b = blockIdx.y;
    const float* q = a.q + (int64_t)b * a.dim;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int first = (blockIdx.x * (kDotThreads / 64) + wave) * kRowsPerWave;
    if (first >= a.max_n) return;
    int item[kRowsPerWave];
    bool ok[kRowsPerWave];
    const float* row[kRowsPerWave];
    float acc[kRowsPerWave];
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r) {
        const int j = first + r < a.max_n ? first + r : a.max_n - 1;
        item[r] = a.idx[(int64_t)b * a.max_n + j];
    }
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r) {
        ok[r] = item[r] >= 0 && item[r] < a.n_items;
        row[r] = a.data + (int64_t)(ok[r] ? item[r] : 0) * a.dim;  // row 0 stands in: always readable
        acc[r] = 0.0f;
    }
    if ((a.dim & 3) == 0) {
        auto chunks = [&](int base, auto n_) {
            constexpr int n = decltype(n_)::value;
            f32x4 x[n][kRowsPerWave];
            f32x4u y[n];
#pragma unroll
            for (int i = 0; i < n; ++i) {
                const int c = base + i * 256 + lane * 4;
                y[i] = *reinterpret_cast<const f32x4u*>(q + c);
#pragma unroll
                for (int r = 0; r < kRowsPerWave; ++r)
                    x[i][r] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(row[r] + c));
            }
#pragma unroll
            for (int i = 0; i < n; ++i)
#pragma unroll
                for (int r = 0; r < kRowsPerWave; ++r) {
                    acc[r] = __builtin_fmaf(x[i][r].x, y[i].x, acc[r]);
                    acc[r] = __builtin_fmaf(x[i][r].y, y[i].y, acc[r]);
                    acc[r] = __builtin_fmaf(x[i][r].z, y[i].z, acc[r]);
                    acc[r] = __builtin_fmaf(x[i][r].w, y[i].w, acc[r]);
                }
        };
        int base = 0;
        for (; base + kDotChunks * 256 <= a.dim; base += kDotChunks * 256) chunks(base, std::integral_constant<int, kDotChunks>{});
        if (base + 512 <= a.dim) {
            chunks(base, std::integral_constant<int, 2>{});
            base += 512;
        }
        if (base + 256 <= a.dim) {
            chunks(base, std::integral_constant<int, 1>{});
            base += 256;
        }
        if (base + lane * 4 < a.dim) chunks(base, std::integral_constant<int, 1>{});
    } else {
        for (int c = lane; c < a.dim; c += 64) {
#pragma unroll
            for (int r = 0; r < kRowsPerWave; ++r) acc[r] = __builtin_fmaf(row[r][c], q[c], acc[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r) {
        const float t = wave_sum_last(acc[r]);
        const int j = first + r;
        if (lane == 63 && j < a.max_n) a.keys[b * key_pitch(a.max_n) + j] = ok[r] ? score_key(t) : 0u;
    }
}

}  // namespace

extern "C" size_t ucm_dot_topk_workspace_bytes(int32_t B, int32_t max_n)
{
    if (B <= 0 || max_n <= 0) return 256;
    return (size_t)B * key_pitch(max_n) * 4;
}

extern "C" int ucm_dot_topk(const float* data, int64_t n_items, int32_t dim, const float* query,
                            const int32_t* indexes, int32_t B, int32_t max_n, int32_t topk,
                            int32_t* out_idx, float* out_score, void* workspace,
                            size_t workspace_bytes, ucm_stream_t stream)
{
    ucm::clear_error();
    UCM_REQUIRE(B >= 0 && B <= 65535, "batch %d out of range [0, 65535]", B);
    if (B == 0) return UCM_OK;
    UCM_REQUIRE(data && query && indexes && out_idx && out_score, "null pointer");
    UCM_REQUIRE(n_items > 0 && dim > 0 && max_n > 0, "non-positive shape");
    UCM_REQUIRE(topk > 0, "topk %d must be positive", topk);
    if (topk > kMaxTopk) return ucm::fail(UCM_EUNSUPPORTED, "topk %d above %d", topk, kMaxTopk);
    UCM_REQUIRE(dim <= 16384, "dim %d above 16384", dim);  // the documented limit; nothing in the kernels depends on it
    UCM_REQUIRE(workspace && workspace_bytes >= ucm_dot_topk_workspace_bytes(B, max_n),
                "workspace too small");
    UCM_REQUIRE((((uintptr_t)data | (uintptr_t)workspace) & 15) == 0, "data must be 16-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    DotArgs d{};
    d.data = data; d.n_items = n_items; d.dim = dim; d.q = query; d.idx = indexes; d.max_n = max_n;
    d.keys = (uint32_t*)workspace;
    const int rows_per_wg = (kDotThreads / 64) * kRowsPerWave;
    hipLaunchKernelGGL(dot_score_kernel, dim3((unsigned)ucm::ceil_div(max_n, rows_per_wg), (unsigned)B),
                       dim3(kDotThreads), 0, st, ucm::arg_pair(d.data, d.q), ucm::arg_pair(d.idx, d.keys),
                       ucm::ArgInts{dim, max_n, (int)(uint32_t)n_items, (int)(n_items >> 32)});
    int rc = ucm::launch_status("dot_score_kernel");
    if (rc != UCM_OK) return rc;
    SortArgs s{};
    s.keys = d.keys; s.idx = indexes; s.max_n = max_n; s.topk = topk;
    s.out_idx = out_idx; s.out_score = out_score;
    return launch_topk(s, B, st);
}
