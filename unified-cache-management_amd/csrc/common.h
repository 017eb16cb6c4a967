// Shared host-side helpers of the HIP library: status codes, per-thread error text,
// HIP error translation.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>

#include "ucm_hip.h"

namespace ucm {

// Stores a printf-formatted message for ucm_last_error() and returns `code`.
int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
void clear_error();

inline int hip_fail(hipError_t e, const char* what)
{
    // hipGetLastError() resets the sticky error so that a later, unrelated call does not
    // report this failure again.
    (void)hipGetLastError();
    return fail(e == hipErrorOutOfMemory ? UCM_EOOM : UCM_ERROR, "%s: %s", what,
                hipGetErrorString(e));
}

#define UCM_HIP_TRY(expr)                                          \
    do {                                                           \
        hipError_t e__ = (expr);                                   \
        if (e__ != hipSuccess) return ::ucm::hip_fail(e__, #expr); \
    } while (0)

#define UCM_REQUIRE(cond, ...)                                        \
    do {                                                              \
        if (!(cond)) return ::ucm::fail(UCM_EPARAM, __VA_ARGS__);     \
    } while (0)

inline int launch_status(const char* kernel)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(UCM_ERROR, "launch of %s failed: %s", kernel, hipGetErrorString(e));
    return UCM_OK;
}

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

#ifdef __HIPCC__
// What a kernel's first loads take goes into leading arguments of these types: the build has the hardware put the first
// fourteen words of scalar and vector arguments into registers before the waves start, where the fields of a struct
// are read from memory by every wave, 0.2 to 0.5 us in front of its first load.  Vectors, as every argument of a launch
// costs the host some 25 ns (two launches with twelve arguments more: 8.6 and 8.9 us a call that waits for its host).
typedef uint64_t ArgPair __attribute__((ext_vector_type(2)));
typedef int32_t ArgInts __attribute__((ext_vector_type(4)));
inline ArgPair arg_pair(const void* a, const void* b) { return ArgPair{(uint64_t)(uintptr_t)a, (uint64_t)(uintptr_t)b}; }
inline ArgPair arg_pair(const void* a, uint64_t b) { return ArgPair{(uint64_t)(uintptr_t)a, b}; }
inline uint64_t arg_words(int lo, int hi) { return (uint32_t)lo | (uint64_t)(uint32_t)hi << 32; }
__device__ __forceinline__ int arg_lo(uint64_t v) { return (int)(uint32_t)v; }
__device__ __forceinline__ int arg_hi(uint64_t v) { return (int)(v >> 32); }
// (by way of the global address space: an address of unknown space would make every access a flat one)
template <class T>
__device__ __forceinline__ T* arg_ptr(uint64_t v)
{
    return (T*)(__attribute__((address_space(1))) T*)v;
}

// Touches every 64-byte line of a kernel-argument struct at once.  The compiler fetches a field
// where the code first needs it, behind the branches of the row addressing - a dozen scalar reads
// one after the other in a kernel that lives for a few microseconds; with the lines already in the
// scalar cache those reads are short.  (Copying the struct through pinned registers instead makes
// its pointers lose their address space: every access becomes a flat one.)
template <class T>
__device__ __forceinline__ void warm_args(const T& args)
{
    const uint32_t* src = reinterpret_cast<const uint32_t*>(&args);
    uint32_t t = 0;
#pragma unroll
    for (unsigned i = 0; i < sizeof(T) / 4; i += 16) t |= src[i];
    t |= src[sizeof(T) / 4 - 1];
    asm volatile("" ::"s"(t));
}
#endif

// hash_encode.hip: one (new keys -> paged cache, queries -> codes) pair of a decode step.
// Strides of keys and queries in elements, of the cache and of q_codes in 32-bit words.
struct PairSpec {
    const void* keys; int64_t T; int Hkv; int64_t k_stride_t, k_stride_h;
    const void* slot; int slot_is_i64;
    uint32_t* cache; int64_t NB; int BS; int64_t cs_block, cs_token, cs_head;
    const void* queries; int64_t B; int Hq; int64_t q_stride_b, q_stride_h;
    uint32_t* q_codes; int64_t qc_stride_b, qc_stride_h;
    int x_dtype; int K; const void* w; int w_dtype; int n_w; int N_bits;
    int q_group_mean = 0;  // hash the mean of every KV head's query group: q_codes is [B, Hkv, Wd]
    // latent attention's head reduction: query row i of the Hq / q_reduce that are hashed is the mean
    // of heads i, i + Hq / q_reduce, i + 2 * Hq / q_reduce, ... (q_codes is [B, Hq / q_reduce, Wd])
    int q_reduce = 0;
};
// The block scores of a grouped-query decode step: best KV head, sink and recent blocks kept (see ucm_hamming_topk).
struct StepScore {
    const int32_t* table; int table_stride, max_blocks; const int32_t* lens; int sink, recent;
    int32_t* scores;  // [B][max_blocks]
};
// whether encode_and_score() takes the step; fails as encode_pair() would
int step_is_fused(const PairSpec& p, const StepScore& s, bool& fused);
// both jobs of a pair and the block scores in one launch
int encode_and_score(const PairSpec& p, const StepScore& s, hipStream_t st);
// one launch when both jobs are small
int encode_pair(const PairSpec& p, hipStream_t st);
// two pairs; one launch when all four jobs are small and the input widths are 512 and 64
int encode_two_pairs(const PairSpec& a, const PairSpec& b, hipStream_t st);

}  // namespace ucm
