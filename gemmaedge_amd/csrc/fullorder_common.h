// What the full-order kernels share (fullorder_kernels.hip, the histogram and
// sort-based passes; fullorder_binned.hip, f32 rows without a sort): which
// rows they serve, the per-row meta words, and when an error interval decides
// what the reference takes from a sequential double sum.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ge_math.h"
#include "sampler_internal.h"

#pragma clang fp contract(off)

namespace ge {
namespace {

enum : uint32_t {
    kMetaItems = 0, kMetaExtras = 1, kMetaNan = 2, kMetaStatus = 3,
    // sorted rows only: the top k's exps, from the sort kernel (their sum
    // as two words of a double, the lowest set bit, any NaN)
    kMetaSumLo = 4, kMetaSumHi = 5, kMetaMinLsb = 6, kMetaAnyNan = 7,
    // f32 calls: the tiles of a left row that are done, and (row 0) the next
    // work item of fo_left_kernel; the sort-free kernels clear both
    kMetaProgress = 8, kMetaTicket = 9
};
// kStatusToSort: a row left to the sort-based fallback pass (bf16: more
// penalised ids than the extras hold; f32: not served without a sort);
// kStatusFallback: items of such a row, made by the fallback sort;
// kStatusSkip: a row the fallback pass leaves as the first pass wrote it.
enum : uint32_t { kStatusOk = 0, kStatusToSort = 1, kStatusFallback = 2, kStatusSkip = 3 };

// generation.cpp:66, :80 — rows this path serves: sampling (T > 0 or NaN) with k > kMaxTopK.
__device__ __forceinline__ bool full_order_row(const ge_sample_params& p, int V, uint32_t& k) {
    if (p.temperature <= 0.0f) return false;
    k = p.top_k ? min(p.top_k, static_cast<uint32_t>(V)) : static_cast<uint32_t>(V);
    return k > static_cast<uint32_t>(kMaxTopK);
}

__device__ __forceinline__ void history_of(const DevArgs& a, int row, const int32_t*& h, int& n) {
    h = nullptr;
    n = 0;
    if (a.ring) {
        h = a.ring + static_cast<int64_t>(row) * a.ring_capacity;
        n = min(max(a.ring_len[row], 0), a.ring_capacity);
    } else if (a.history && a.history_offsets) {
        const int s = a.history_offsets[row];
        h = a.history + s;
        n = max(a.history_offsets[row + 1] - s, 0);
    }
}

__device__ __forceinline__ int exp_of(double d) {  // floor(log2 d), d > 0 normal
    return static_cast<int>((__builtin_bit_cast(uint64_t, d) >> 52) & 0x7ff) - 1023;
}

// Buffer reads of the sort read from L2 (agent-scope loads skip the CU's L1),
// so a line the L1 kept from an earlier pass is never used after another wave
// of the workgroup rewrote it; the writers wait for their stores before each
// barrier.
__device__ __forceinline__ uint32_t ld_l2(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The exponent whose binade holds the sequential sum that S approximates (the
// two differ by far less than 2^-20), or the one above.
__device__ __forceinline__ int sum_exp(double S) { return exp_of(S * (1.0 + 0x1p-20)); }

// Whether the reciprocal 1 / den rounds to the same float for every value that
// the reference's sequential double sum can have, S being a sum of the same
// terms in another order: then no replay is needed, as only that float is
// used (generation.cpp:98-101). With e = sum_exp(S) and U = 2^(e-52), a term
// whose lowest set bit is at least U adds without rounding except where the
// sum enters a higher binade (the sum starts at exp(0) = 1, so at most e
// times); a float at or above 2^(e-29) is such a term. Each other term
// (`fine` of them, or more) rounds by at most U / 2. The parallel sum adds at
// most V / 512 + 512 roundings of at most U in sequence. The interval so
// bounded straddles a rounding boundary of the float for about one row in
// 10^4 to 10^3 (26,000 to 262,144 fine terms); those are replayed. Before,
// every row whose terms span more than 53 bits was (sigma-3 logits,
// V = 262,144): 48 bf16 rows of which 8 are full order 324 -> 151 us a call, one
// f32 row 245 -> 203 us, 64 f32 rows 828 -> 634 us.
__device__ __forceinline__ bool den_rounds_alike(double S, uint32_t fine, int V) {
    if (!(S >= 0.5) || !(S < 0x1p60)) return false;
    const double eps = (static_cast<double>(fine) + 64.0 + 2.0 * (static_cast<double>(V) / 512.0 + 512.0)) *
                       __builtin_ldexp(1.0, sum_exp(S) - 53) * (1.0 + 0x1p-10);
    return static_cast<float>(1.0 / (S - eps)) == static_cast<float>(1.0 / (S + eps));
}

// How far two double sums of `n` probabilities in different orders, and of one
// term more, can lie apart (the sums are below 2: at most 2^-53 a rounding).
__device__ __forceinline__ double near_sum_error(uint32_t n) { return (2.0 * n + 16.0) * 0x1p-53 * (1.0 + 0x1p-10); }

// Whether |x - c| < 1e-6 is decided for every c within eps of `c`; `near` is
// its value then.
__device__ __forceinline__ bool near_decided(double x, double c, double eps, bool& near) {
    const double d = __builtin_fabs(x - c);
    near = d < 1e-6;
    return d <= 1e-6 - eps || d >= 1e-6 + eps;
}


// First index in [lo, hi) whose predicate is false, for a predicate that is
// true on a prefix; 64-way search with one wave.
template <typename Pred>
__device__ uint32_t wave_partition_point(uint32_t lo, uint32_t hi, Pred pred) {
    const int lane = __lane_id();
    while (hi > lo) {
        const uint32_t step = (hi - lo + 63) / 64;
        const uint32_t probe = lo + static_cast<uint32_t>(lane) * step;
        const uint64_t m = __ballot(probe < hi && pred(probe));
        if (m == 0) break;  // pred(lo) is false
        const int last = 63 - static_cast<int>(__builtin_clzll(m));
        lo = lo + static_cast<uint32_t>(last) * step + 1;
        hi = min(hi, lo - 1 + step);
    }
    return lo;
}

}  // namespace
}  // namespace ge
