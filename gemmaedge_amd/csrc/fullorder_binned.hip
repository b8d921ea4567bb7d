// Full-order sampling of f32 rows without a sort (top-k disabled: k = V,
// src/generation.cpp:80).
//
// The reference sorts the row and then adds the probabilities one by one in
// float: the top-p cumulative, and the draw's subtract walk. Inside one
// binade of the accumulator such a sum moves by whole ulps, and the number of
// ulps that an addend q adds, round(q / ulp), does not depend on the order
// (chain_math.h; an exact tie does, through the accumulator's parity). So the
// order only matters where the accumulator changes binade, where an addend
// ties, and where the sum stops. The row is therefore cut into bins of
// neighbouring probabilities: where all of a bin's addends round alike it is a
// count times an integer, where they do not its tokens' integers are summed,
// and only the bins with a binade change, a tie or a stop (a few thousand
// tokens of a near-uniform row of V = 262,144) are sorted and taken one by one.
//
//   fb_range    marks the history ids; the row's largest final value and
//               smallest raw one
//   fb_exps     every token's exp((v - max) / T), kept; their sum; their
//               histogram in bins of equal width in the float's bits
//   fb_plan     1 / denominator; per bin the probabilities' sum before it and
//               the walk's, following the float sums' rounding; the ulps of the
//               bins whose addends round alike; which bins are expanded into
//               tokens, and which of those the chains replay
//   fb_collect  the expanded bins' tokens; the sum of the probabilities
//               before the bins the draw can end in
//   fb_order    the expanded bins' ulps, or their tokens in order
//   fb_draw     the chains, the token, and a check that the bins between two
//               replayed ones were passed in the binade the plan took them in
//
// Results are exact for any plan: fb_draw checks over every gap between
// replayed bins that the sums had the binade which the plan took the gap in,
// and otherwise leaves the row to the sort, as the plan leaves rows that this
// path does not serve (NaN or infinite maxima, a denominator whose reciprocal
// the sum's error interval leaves open, replayed bins of more than kFbSegMost
// tokens, more replayed tokens than the draw's lists hold). Of 2,048 rows each
// at V = 32,003 to 262,144, T 0.6 to 1.3 and top_p 0.9 to 2: none of near-uniform
// ones, 0 to 12 of normal (sigma 3), Zipf, confident and masked ones (35 at T 1.3,
// top_p 1, V = 262,144), up to 350 of logits on a grid of 1/8.
//
// Measured against the radix sort it replaces (whole calls, V = 262,144): one
// row 241 -> 97 us, 64 rows 822 -> 185 us, 512 near-uniform rows 4,820 ->
// 1,063 us; of the last, per 256 rows: range 64, exps 171, plan 57, collect 92,
// order 66, draw 81 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <type_traits>

#include "chain_math.h"
#include "fullorder_common.h"
#include "ge_math.h"
#include "sampler_internal.h"
#include "wave_ops.h"

#pragma clang fp contract(off)

namespace ge {
namespace {

constexpr int kFT = 1024;              // threads of the streaming kernels and the plan
constexpr int kFW = kFT / 64;
constexpr int kFStep = kFT * 4;        // tokens of one 16-byte load per thread
constexpr uint32_t kOne = 0x3f800000u; // the bits of 1.0f, the largest exp
constexpr uint32_t kLeast = 0x2f800000u;  // 2^-32: where the bins' width stops following the smallest exp
constexpr uint32_t kFbHead = 1024;     // tokens always expanded
constexpr int kFbWaveSeg = 512;        // tokens of a bin that one wave orders
constexpr uint32_t kFbSegMost = 4096;  // tokens of an expanded bin at most
constexpr double kFbDrift = 0x1p-14;   // the plan's relative margin on a float sum

// One expanded bin. What the chains add (cumulative) or take off (walk) for the
// bins between two replayed ones is a sum of whole ulps of one binade.
struct FbSeg {
    uint32_t item;    // its tokens' first item
    uint32_t n;       // its tokens
    uint32_t elem;    // its first element (the tokens before it)
    uint32_t info;    // biased exponents of the two accumulators before it, and kSeg* flags
    double cum;       // ulps that the unexpanded bins before it add to the cumulative
    double walk;      // ulps that they take off in the walk
    uint32_t scum;    // ulps that this bin's own tokens add, when it is not replayed
    uint32_t swalk;
};
static_assert(sizeof(FbSeg) == 4 * kFbSegWords, "the area's size");
enum : uint32_t {
    kSegReplayCum = 1u << 16,   // the cumulative takes its tokens one by one
    kSegReplayWalk = 1u << 17,  // the walk does
    kSegInWalk = 1u << 18       // the walk may reach it
};

// The row's area in fo_tiles.
struct FbRow {
    uint32_t* bin;    // [bins] counts, then the expanded bins' next item
    uint32_t* pmax;   // [kFbParts] largest final key
    uint32_t* pmin;   // [kFbParts] smallest raw key
    double* psum;     // [kFbParts] sums of exps
    double* pbef;     // [kFbParts] sums of the probabilities before the draw's bins
    uint32_t* scal;   // [kScalWords]
    uint32_t* mask;   // [bins / 32] expanded bins
    FbSeg* seg;       // [kFbSegs + 1] the expanded bins, in order, and the list's end
};
// (kScLarge: fb_order met a bin too large to order, so the draw leaves the row)
enum : int { kScShift = 0, kScInv, kScDrawBin, kScDrawItem, kScDrawEnd, kScSegs, kScCut, kScLarge, kScalWords = 64 };

__device__ __forceinline__ FbRow fb_row(const DevArgs& a, int row, int bins) {
    uint32_t* w = a.fo_tiles + static_cast<int64_t>(row) * fb_row_words(a.vocab);
    FbRow r;
    r.bin = w;
    r.pmax = w + bins;
    r.pmin = r.pmax + kFbParts;
    r.psum = reinterpret_cast<double*>(r.pmin + kFbParts);
    r.pbef = r.psum + kFbParts;
    r.scal = reinterpret_cast<uint32_t*>(r.pbef + kFbParts);
    r.mask = r.scal + kScalWords;
    r.seg = reinterpret_cast<FbSeg*>(r.mask + kFbMaxBins / 32);
    return r;
}
// The row's exps.
__device__ __forceinline__ float* fb_exp_array(const DevArgs& a, int row) {
    return a.fo_aux + static_cast<int64_t>(row) * a.fo_items_stride;
}
__device__ __forceinline__ uint32_t fb_bin(float pe, uint32_t shift, uint32_t bins) {
    return min((kOne - f2u(pe)) >> shift, bins - 1u);
}
// Rows this path serves: sampling rows with k = V.
__device__ __forceinline__ bool fb_serves(const DevArgs& a, int row, ge_sample_params& p) {
    p = a.row_params ? a.row_params[row] : a.params;
    uint32_t k;
    return full_order_row(p, a.vocab, k) && !row_done(a, row) && k == static_cast<uint32_t>(a.vocab);
}
__device__ __forceinline__ uint32_t* fb_meta(const DevArgs& a, int row) {
    return a.fo_meta + static_cast<int64_t>(row) * kMetaWords;
}
// Tokens [lo, hi) of a part: whole steps of kFStep.
__device__ __forceinline__ void fb_part(const DevArgs& a, int part, int parts, int& lo, int& hi) {
    const int steps = (a.vocab + kFStep - 1) / kFStep;
    const int per = (steps + parts - 1) / parts * kFStep;
    lo = min(part * per, a.vocab);
    hi = min(lo + per, a.vocab);
}

// f(token, x0, x1, x2, x3, tokens valid) over [lo, hi) in steps of kU 16-byte
// loads per thread; rows that are not 16-byte aligned load single values.
template <int kU, typename F>
__device__ __forceinline__ void fb_stream(const float* rowp, bool vec, int lo, int hi, int tid, F&& f) {
    typedef float v4 __attribute__((ext_vector_type(4)));
    int base = lo;
    if (vec) {
        for (; base + kU * kFStep <= hi; base += kU * kFStep) {
            v4 x[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) x[u] = *reinterpret_cast<const v4*>(rowp + base + u * kFStep + tid * 4);
#pragma unroll
            for (int u = 0; u < kU; ++u) f(base + u * kFStep + tid * 4, x[u].x, x[u].y, x[u].z, x[u].w, 4);
        }
    }
    for (; base < hi; base += kFStep) {
        const int i = base + tid * 4;
        float x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = rowp[min(i + j, hi - 1)];  // clamped: no conditional load
        f(i, x[0], x[1], x[2], x[3], min(max(hi - i, 0), 4));
    }
}

// f(first token, x[kU][4], tokens from it on): one call per step of kU 16-byte
// loads per thread, load u at first + u * kFStep; the last step may be partial
// (tokens past the end repeat the last one).
template <int kU, typename F>
__device__ __forceinline__ void fb_stream_steps(const float* rowp, bool vec, int lo, int hi, int tid, F&& f) {
    typedef float v4 __attribute__((ext_vector_type(4)));
    for (int base = lo; base < hi; base += kU * kFStep) {
        float x[kU][4];
        const int i0 = base + tid * 4;
        if (vec && base + kU * kFStep <= hi) {
            v4 q[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) q[u] = *reinterpret_cast<const v4*>(rowp + i0 + u * kFStep);
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                x[u][0] = q[u].x;
                x[u][1] = q[u].y;
                x[u][2] = q[u].z;
                x[u][3] = q[u].w;
            }
        } else {
#pragma unroll
            for (int u = 0; u < kU; ++u)
#pragma unroll
                for (int j = 0; j < 4; ++j) x[u][j] = rowp[min(i0 + u * kFStep + j, hi - 1)];
        }
        f(i0, x, base + kU * kFStep <= hi ? kU * kFStep : hi - i0);
    }
}

// The words that fo_left_kernel counts in, for any row of the call (one thread).
__device__ __forceinline__ void fb_clear_left(const DevArgs& a, int row) {
    fb_meta(a, row)[kMetaProgress] = 0u;
    if (row == 0) fb_meta(a, row)[kMetaTicket] = 0u;
}

// Largest and smallest of one key per thread over the workgroup.
__device__ __forceinline__ uint32_t fb_block_max(uint32_t v, uint32_t* s) {
    const uint32_t w = wave::max_u32(v);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = w;
    __syncthreads();
    uint32_t m = 0;
    for (int i = 0; i < kFW; ++i) m = max(m, s[i]);
    __syncthreads();
    return m;
}

// 1. The part's history bits, its largest final key and smallest raw key.
//    A streaming read: bound by memory at many rows, by latency at few.
struct RangeShared {
    uint32_t s[kFW];
};
__device__ __forceinline__ void fb_range(const DevArgs& a, int row, int part, int parts, RangeShared& sh) {
    uint32_t* s = sh.s;
    const int tid = threadIdx.x;
    ge_sample_params p;
    const int bins = a.fo_bins;
    if (!fb_serves(a, row, p)) {
        uint32_t k;
        // (a row of this pass that the sort-based one serves: 1024 < k < V)
        if (part == 0 && tid == 0 && full_order_row(p, a.vocab, k) && !row_done(a, row))
            fb_meta(a, row)[kMetaStatus] = kStatusToSort;
        return;
    }
    const FbRow r = fb_row(a, row, bins);
    for (int i = part * kFT + tid; i < bins; i += parts * kFT) r.bin[i] = 0u;
    int lo, hi;
    fb_part(a, part, parts, lo, hi);
    const int32_t* hist;
    int H;
    history_of(a, row, hist, H);
    const bool pen = H > 0 && !(p.repetition_penalty == 1.0f);
    const float* rowp = static_cast<const float*>(a.logits) + static_cast<int64_t>(row) * a.row_stride;
    uint32_t* bitmap = a.fo_bitmap + static_cast<int64_t>(row) * a.fo_bitmap_words;
    uint32_t top = 0u;
    if (pen) {
        for (int i = tid; i < H; i += kFT) {
            const int32_t id = hist[i];
            if (id >= lo && id < hi) {
                atomicOr(&bitmap[id >> 5], 1u << (id & 31));
                top = max(top, order_key(penalize(softcap(rowp[id], p.softcap), p.repetition_penalty)));
            }
        }
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
    }
    float mx = NAN, mn = NAN;
    fb_stream<4>(rowp, a.vec_ok != 0, lo, hi, tid, [&](int i, float x0, float x1, float x2, float x3, int n) {
        const uint32_t bits = pen && n ? ld_l2(bitmap + (i >> 5)) >> (i & 31) : 0u;
        const float x[4] = {x0, x1, x2, x3};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (j < n) {
                mn = fminf(mn, x[j]);
                if (!((bits >> j) & 1u)) mx = fmaxf(mx, x[j]);
            }
        }
    });
    // (NaN: no number seen; keys 0 and all ones then)
    const uint32_t kx = fb_block_max(mx == mx ? order_key(mx) : 0u, s);
    const uint32_t kn = ~fb_block_max(mn == mn ? ~order_key(mn) : 0u, s);
    const uint32_t kt = fb_block_max(top, s);
    if (tid == 0) {
        r.pmax[part] = max(kt, kx != 0u ? order_key(softcap(key_value(kx), p.softcap)) : 0u);
        r.pmin[part] = kn;
    }
}

// The row's largest final value and the bins' width: the exps of the row,
// from 1 down to the smallest one (2^-32 at least), over all bins. The width is a
// power of two of the float's bits: for a row down to 2^-32 its 2^28 bits take
// half the bins, and the other half reaches 2^-64, below which the exps share
// the last bin. (Bins half as wide could be twice kFbSegs when all are expanded.)
__device__ __forceinline__ void fb_bin_shape(const FbRow& r, int parts, int bins, const ge_sample_params& p, float& vmax,
                                             uint32_t& shift) {
    const int lane = __lane_id();
    const uint32_t kx = wave::max_u32(lane < parts ? r.pmax[lane] : 0u);
    const uint32_t kn = wave::min_u32(lane < parts ? r.pmin[lane] : 0xffffffffu);
    vmax = key_value(kx);
    const float pe = expf_glibc((softcap(key_value(kn), p.softcap) - vmax) * (1.0f / p.temperature));
    const uint32_t low = pe >= u2f(kLeast) && pe <= 1.0f ? f2u(pe) : kLeast;
    const int len = 32 - __clz(static_cast<int>(kOne - low));  // (0 when every exp is 1)
    shift = static_cast<uint32_t>(max(len - (31 - __clz(bins)), 0));
}

// 2. Each token's exp (generation.cpp:94-97: exp((l - max) * (1 / T)), of the
//    capped and penalised value), the part's sum of them, and the histogram of
//    their bins. Bound by the exact tanhf and expf (about 130 instructions a
//    token), which a step's 16 tokens per thread overlap.
struct ExpsShared {
    uint32_t hist[kFbMaxBins];
    uint64_t tab[32];
    double sums[kFW];
    float vmax;
    uint32_t shift;
};
__device__ __forceinline__ void fb_exps(const DevArgs& a, int row, int part, int parts, ExpsShared& sh) {
    uint32_t* hist_s = sh.hist;
    uint64_t* tab = sh.tab;
    double* sums = sh.sums;
    const int tid = threadIdx.x;
    ge_sample_params p;
    if (!fb_serves(a, row, p)) return;
    const int bins = a.fo_bins;
    const FbRow r = fb_row(a, row, bins);
    if (tid < 64) {
        float vm;
        uint32_t sf;
        fb_bin_shape(r, parts, bins, p, vm, sf);
        if (tid == 0) {
            sh.vmax = vm;
            sh.shift = sf;
        }
        if (tid < 32) tab[tid] = exp2_table(static_cast<uint32_t>(tid));
    }
    for (int i = tid; i < bins; i += kFT) hist_s[i] = 0u;
    __syncthreads();
    const float vmax = sh.vmax;
    const uint32_t shift = sh.shift;
    int lo, hi;
    fb_part(a, part, parts, lo, hi);
    const int32_t* hist;
    int H;
    history_of(a, row, hist, H);
    const bool pen = H > 0 && !(p.repetition_penalty == 1.0f);
    const float* rowp = static_cast<const float*>(a.logits) + static_cast<int64_t>(row) * a.row_stride;
    const uint32_t* bitmap = a.fo_bitmap + static_cast<int64_t>(row) * a.fo_bitmap_words;
    float* pes = fb_exp_array(a, row);
    const float inv_temp = 1.0f / p.temperature;
    const float cap = p.softcap;
    // The narrow softcaps apply to a step whose logits all lie in their range
    // (one vote per 16 tokens a lane). Below 2^-100 * cap the quotients may round
    // otherwise, which no exp shows unless 1 / T is huge.
    const bool capped = cap > 0.0f;
    const bool narrow = capped && cap >= 0x1p-60f && cap <= 0x1p60f && inv_temp <= 0x1p40f;
    const float small = narrow ? cap * kSoftcapSmall : -1.0f, below = narrow ? cap * kSoftcapBelowOne : -1.0f;
    const float yc = narrow ? recip_step(cap) : 0.0f;
    double sum = 0.0;
    fb_stream_steps<4>(rowp, a.vec_ok != 0, lo, hi, tid, [&](int i0, const float (&x)[4][4], int n) {
        float most = 0.0f;
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int j = 0; j < 4; ++j) most = fmaxf(most, __builtin_fabsf(x[u][j]));
        auto take = [&](auto&& cap_of) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = i0 + u * kFStep;
                const int nu = min(max(n - u * kFStep, 0), 4);
                if (n < 4 * kFStep && nu == 0) continue;
                const uint32_t bits = pen ? bitmap[i >> 5] >> (i & 31) : 0u;
                float pe[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float v = cap_of(x[u][j]);
                    if ((bits >> j) & 1u) v = penalize(v, p.repetition_penalty);
                    pe[j] = expf_glibc_tab((v - vmax) * inv_temp, [&](uint32_t t) { return tab[t]; });
                }
                if (n >= 4 * kFStep || nu == 4) {
                    *reinterpret_cast<float4*>(pes + i) = make_float4(pe[0], pe[1], pe[2], pe[3]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        sum += static_cast<double>(pe[j]);
                        atomicAdd(&hist_s[fb_bin(pe[j], shift, static_cast<uint32_t>(bins))], 1u);
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        if (j < nu) {
                            pes[i + j] = pe[j];
                            sum += static_cast<double>(pe[j]);
                            atomicAdd(&hist_s[fb_bin(pe[j], shift, static_cast<uint32_t>(bins))], 1u);
                        }
                    }
                }
            }
        };
        if (!capped) take([&](float v) { return v; });
        else if (__ballot(!(most <= small)) == 0ull) take([&](float v) { return softcap_range<kSoftcapRangeSmall>(v, cap, yc); });
        else if (__ballot(!(most <= below)) == 0ull) take([&](float v) { return softcap_range<kSoftcapRangeBelowOne>(v, cap, yc); });
        else take([&](float v) { return softcap(v, cap); });
    });
    sum = wave::sum_f64(sum);
    if ((tid & 63) == 0) sums[tid >> 6] = sum;
    __syncthreads();
    if (tid == 0) {
        double t = 0.0;
        for (int w = 0; w < kFW; ++w) t += sums[w];
        r.psum[part] = t;
    }
    // (two bins per word: the counts do not reach 2^32)
    unsigned long long* out = reinterpret_cast<unsigned long long*>(r.bin);
    for (int i = tid; i < bins / 2; i += kFT) {
        const unsigned long long c = (static_cast<unsigned long long>(hist_s[2 * i + 1]) << 32) | hist_s[2 * i];
        if (parts == 1) out[i] = c;
        else if (c) atomicAdd(&out[i], c);
    }
}

// Exclusive prefix of one double (count) per thread over the workgroup, and
// the total. The order of the additions is fixed.
template <int kWaves>
__device__ __forceinline__ double fb_scan_f64(double v, double* s, double& total) {
    const int wave = threadIdx.x >> 6;
    const double incl = wave::incl_f64(v);
    if ((threadIdx.x & 63) == 63) s[wave] = incl;
    __syncthreads();
    double before = 0.0;
    total = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        if (w == wave) before = total;
        total += s[w];
    }
    __syncthreads();
    return before + (incl - v);
}
// The same for two counts and a double at once: v, w and x become their
// exclusive prefixes.
template <int kWaves>
__device__ __forceinline__ void fb_scan_3(uint32_t& v, uint32_t& w, double& x, double* sx, uint32_t* sv, uint32_t* sw,
                                          uint32_t& v_all, uint32_t& w_all, double& x_all) {
    const int wave = threadIdx.x >> 6;
    const uint32_t iv = wave::incl_add(v), iw = wave::incl_add(w);
    const double ix = wave::incl_f64(x);
    if ((threadIdx.x & 63) == 63) {
        sv[wave] = iv;
        sw[wave] = iw;
        sx[wave] = ix;
    }
    __syncthreads();
    uint32_t bv = 0, bw = 0;
    double bx = 0.0;
    v_all = w_all = 0;
    x_all = 0.0;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) {
        if (i == wave) {
            bv = v_all;
            bw = w_all;
            bx = x_all;
        }
        v_all += sv[i];
        w_all += sw[i];
        x_all += sx[i];
    }
    __syncthreads();
    v = bv + iv - v;
    w = bw + iw - w;
    x = bx + (ix - x);
}

// The biased float exponent of x > 0, at least 1 (subnormal floats share the
// first normal binade's ulp); 0 for x <= 0.
__device__ __forceinline__ int fb_expo(double x) {
    const int e = static_cast<int>(__builtin_bit_cast(uint64_t, x) >> 52) - 1023 + 127;
    return x > 0.0 ? max(e, 1) : 0;
}
// Whether every addend of [lo, hi] adds the same whole number `n` of ulps in
// the binade with biased exponent e (ulp 2^(e - 150)), none of them a tie.
// (Scaling by a power of two and, below 2^22, adding 1/2 are exact.)
__device__ __forceinline__ bool fb_alike(float lo, float hi, int e, uint32_t& n) {
    const float yl = __builtin_ldexpf(lo, 150 - e), yh = __builtin_ldexpf(hi, 150 - e);
    const float f = __builtin_floorf(yh + 0.5f);
    const bool ok = yh < 0x1p22f && yl > f - 0.5f && yh < f + 0.5f;
    n = ok ? static_cast<uint32_t>(f) : 0u;
    return ok;
}

// 3. One workgroup per row; thread t holds bins kPer * t .., which stay in LDS
//    (kept in registers, 16 bins a thread spill: one row 88 us instead of 36).
//    Bound by its sweeps over the bins on one CU.
struct PlanShared {
    uint32_t c[kFbMaxBins + kFbMaxBins / 16];  // counts (padded: a thread's bins lie 17 words from the next's)
    uint32_t w[kFbMaxBins + kFbMaxBins / 16];  // the bin's rounded sum (a float), then what it is
    double sd[kFW];
    uint32_t su[kFW], sv[kFW];
    uint32_t mask[kFbMaxBins / 32];
    uint32_t bad, cut, cut_elem, stop, first, last, off0, off1;
    double cut_lo, cut_hi;
    float stop_q;
};
template <int kPer>
__device__ __forceinline__ void fb_plan(const DevArgs& a, int row, int parts, PlanShared& sh) {
    constexpr int kBins = kPer * kFT;
    const int tid = threadIdx.x, lane = __lane_id();
    ge_sample_params p;
    if (!fb_serves(a, row, p)) return;
    const int V = a.vocab;
    const FbRow r = fb_row(a, row, kBins);
    uint32_t* meta = fb_meta(a, row);
    const int b0 = tid * kPer;
    auto at_bin = [](int b) { return b + (b >> 4); };
    for (int i = tid; i < kBins; i += kFT) sh.c[at_bin(i)] = r.bin[i];
    float vmax;
    uint32_t shift;
    fb_bin_shape(r, parts, kBins, p, vmax, shift);
    const double S = wave::sum_f64(lane < parts ? r.psum[lane] : 0.0);
    if (tid == 0) {
        sh.bad = 0u;
        sh.cut = sh.cut_elem = sh.stop = sh.first = 0xffffffffu;
        sh.last = 0u;
        sh.cut_lo = sh.cut_hi = 0.0;
        sh.stop_q = 0.0f;
        sh.off0 = sh.off1 = 0u;
    }
    for (int i = tid; i < kBins / 32; i += kFT) sh.mask[i] = 0u;
    __syncthreads();
    const float inv = static_cast<float>(1.0 / S);
    const float minimum = inv * p.min_p;  // generation.cpp:104, probs[0] = 1 * inv
    const double tp = p.top_p == p.top_p ? static_cast<double>(p.top_p) : 1e30;
    const float tiny = S >= 0.5 && S < 0x1p60 ? __builtin_ldexpf(1.0f, min(sum_exp(S) - 29, 0)) : 1.0f;
    // The exps of bin b: [lo_bits, hi_bits] (the last bin: from 0).
    auto hi_pe = [&](int b) { return u2f(kOne - (static_cast<uint32_t>(b) << shift)); };
    auto lo_pe = [&](int b) { return b == kBins - 1 ? 0.0f : u2f(kOne - (static_cast<uint32_t>(b + 1) << shift) + 1u); };
    auto mid = [&](int b) { return 0.5f * (lo_pe(b) * inv + hi_pe(b) * inv); };
    // Bin b's addends in the binade of acc: their mean number of ulps, taken as
    // evenly spread over the bin (rounding its middle instead drifts by 1e-4 over
    // the bins whose addends differ by about half an ulp).
    auto rounded = [&](int b, float c, double acc) {
        const int e = max(fb_expo(acc), 64);  // (below 2^-63 nothing rounds)
        const float yl = __builtin_ldexpf(lo_pe(b) * inv, 150 - e), yh = __builtin_ldexpf(hi_pe(b) * inv, 150 - e);
        const float nl = __builtin_rintf(yl), nh = __builtin_rintf(yh), span = yh - yl;
        float y = nl;
        if (nl != nh) y = span > 1.0f || yh > 4096.0f ? 0.5f * (yl + yh) : nl + (yh - (nh - 0.5f)) / span * (nh - nl);
        return c * __builtin_ldexpf(y, e - 150);
    };
    // f(bin, its padded index, its count) for this thread's bins that hold any.
    auto each = [&](auto&& f) {
        constexpr int kBatch = kPer < 4 ? kPer : 4;
#pragma unroll 1
        for (int j = 0; j < kPer; j += kBatch) {
            uint32_t c[kBatch];
#pragma unroll
            for (int v = 0; v < kBatch; ++v) c[v] = sh.c[at_bin(b0 + j + v)];
#pragma unroll
            for (int v = 0; v < kBatch; ++v)
                if (c[v] != 0u) f(b0 + j + v, at_bin(b0 + j + v), c[v]);
        }
    };
    uint32_t fine = 0, n_t = 0;
    double t = 0.0;
    uint32_t low = 0xffffffffu;  // the min-p cut lies in the first bin with a probability below it
    each([&](int b, int, uint32_t c) {
        n_t += c;
        if (lo_pe(b) < tiny) fine += c;
        if (lo_pe(b) * inv < minimum) low = min(low, static_cast<uint32_t>(b));
        t += static_cast<double>(static_cast<float>(c) * mid(b));
    });
    if (low != 0xffffffffu) atomicMin(&sh.cut, low);
    // one scan for the elements before this thread's bins, the fine terms' number
    // and the exact sum (x)
    uint32_t before = n_t, n_f = fine, total, n_fine;
    double x = t, all;
    fb_scan_3<kFW>(before, n_f, x, sh.sd, sh.su, sh.sv, total, n_fine, all);
    const float inv_temp = 1.0f / p.temperature;
    const bool fits = inv_temp > 0.0f && inv_temp < __builtin_inff() && vmax > -__builtin_inff() &&
                      vmax < __builtin_inff() && total == static_cast<uint32_t>(V) && den_rounds_alike(S, n_fine, V);
    if (!fits) {  // block-uniform
        if (tid == 0) meta[kMetaStatus] = kStatusToSort;
        return;
    }
    // The float sum before each bin: the exact sum first (x), for the binades,
    // then with every addend rounded as it is there (A). The bins' middles miss
    // the exact sum mostly where few large addends hold most of it, in the head
    // (always replayed): the bins after it begin that much later.
    const double corr = S * static_cast<double>(inv) - all;
    x += corr;
    t = 0.0;
    each([&](int b, int i, uint32_t c) {
        const double m = static_cast<double>(static_cast<float>(c) * mid(b));
        const float g = rounded(b, static_cast<float>(c), x + 0.5 * m);
        sh.w[i] = f2u(g);
        t += static_cast<double>(g);
        x += m;
    });
    const double a0 = corr + fb_scan_f64<kFW>(t, sh.sd, all);
    all += corr;
    // f(bin, index, count, the sum before the bin, the sum after it)
    auto sweep = [&](auto&& f) {
        double A = a0;
        each([&](int b, int i, uint32_t c) {
            const double A1 = A + static_cast<double>(u2f(sh.w[i]));
            f(b, i, c, A, A1);
            A = A1;
        });
    };
    const uint32_t cut = sh.cut;  // (written before the scans' barriers)
    sweep([&](int b, int, uint32_t, double A, double A1) {
        if (static_cast<uint32_t>(b) == cut) {
            sh.cut_lo = A;
            sh.cut_hi = A1;
        }
        if (A1 * (1.0 + kFbDrift) >= tp && A * (1.0 + kFbDrift) < tp) atomicMin(&sh.stop, static_cast<uint32_t>(b));
    });
    if (cut == 0xffffffffu && tid == 0) sh.cut_lo = sh.cut_hi = all;
    __syncthreads();
    // The mass the draw is taken of: top_p and less than the stopping addend
    // more, or the sum before the cut; at least the first probability.
    const double q_first = static_cast<double>(inv);
    double mass_lo = tp < sh.cut_lo ? tp : sh.cut_lo;
    const uint32_t stop = sh.stop;
    const double over = tp + (stop != 0xffffffffu ? static_cast<double>(hi_pe(static_cast<int>(stop)) * inv) : 0.0);
    double mass_hi = over < sh.cut_hi ? over : sh.cut_hi;
    if (!(mass_lo > q_first)) {
        mass_lo = q_first;
        mass_hi = max(mass_hi, 2.0 * q_first);
    }
    // (never more than the row holds: twice a first probability near 1 would
    // put the whole tail into the draw's range)
    mass_hi = min(mass_hi, max(all, q_first) * (1.0 + kFbDrift));
    const double u = static_cast<double>(a.uniforms[row]);
    // (a sum that top_p stops is the float itself: only one that ends at the cut
    // or the row's end has drifted)
    const double c_lo = u * mass_lo * (1.0 - (mass_lo < tp ? kFbDrift : 0x1p-20));
    const double c_hi = u * mass_hi * (1.0 + (mass_hi < tp ? kFbDrift : 0x1p-20));
    const double c_mid = 0.5 * (c_lo + c_hi);
    // What the walk has taken off before each bin.
    // (threads whose bins no chain reaches have nothing more to find)
    const bool live = n_t != 0u && (before < kFbHead || (a0 * (1.0 - kFbDrift) < tp && static_cast<uint32_t>(b0) <= cut));
    t = 0.0;
    if (live) sweep([&](int b, int, uint32_t c, double A, double A1) {
        t += static_cast<double>(rounded(b, static_cast<float>(c), c_mid - 0.5 * (A + A1)));
    });
    double W = corr + fb_scan_f64<kFW>(t, sh.sd, all);
    // What each bin is: seen by the chains, expanded, replayed. A seen bin's
    // word then holds its record's info when it is expanded, else the ulps it
    // adds per addend (24 bits) and the walk's exponent.
    uint32_t n_items = 0, n_seg = 0, n_elem = 0;
    double s_cum = 0.0, s_walk = 0.0;  // the unexpanded bins' ulps
    uint32_t at = before;
    uint32_t seen = 0;  // how many of this thread's bins with tokens are (a prefix of them)
    uint32_t expo_end = 0;
    const int e_first = fb_expo(q_first);
    // The walk's ulps per addend of an unexpanded bin.
    auto walk_ulps = [&](int b, int ew) -> uint32_t {
        return ew ? static_cast<uint32_t>(__builtin_floorf(__builtin_ldexpf(hi_pe(b) * inv, 150 - ew) + 0.5f)) : 0u;
    };
    if (live) sweep([&](int b, int i, uint32_t c, double A, double A1) {
        const double W1 = W + static_cast<double>(rounded(b, static_cast<float>(c), c_mid - 0.5 * (A + A1)));
        const bool head = at < kFbHead;
        const double a_lo = A * (1.0 - kFbDrift), a_hi = A1 * (1.0 + kFbDrift);
        const float qh = hi_pe(b) * inv, ql = lo_pe(b) * inv;
        const int ea = fb_expo(a_lo);
        // Addends below half an ulp of the least binade that the sum can be in
        // (it holds the first probability at least) add nothing, in any order
        // and whatever the sum: it neither changes binade nor stops there. So
        // masked tokens and the tail of an open nucleus need no replay, however
        // many they are; every later bin is such a one too.
        const bool none = __builtin_ldexpf(qh, 150 - max(ea, e_first)) < 0.5f;
        // (the cut's bin: only where its tokens lie on both sides of the cut)
        const bool split = static_cast<uint32_t>(b) == cut && qh >= minimum;
        const bool kept = static_cast<uint32_t>(b) < cut || split;
        if (static_cast<uint32_t>(b) == cut) sh.cut_elem = at + (split ? c : 0u);
        if ((head && !none) || ((head || a_lo < tp) && kept)) {
            const bool edge = none ? split : head || split || a_hi >= tp;
            uint32_t dc = 0, dw = 0;
            const bool rc = edge || (!none && (ea != fb_expo(a_hi) || ea == 0));
            bool ex = rc || (!none && !fb_alike(ql, qh, ea, dc));
            int ew = 0;
            bool rw = false;
            const double slack = c_hi * kFbDrift + (head && !none ? __builtin_fabs(corr) : 0.0);
            const double w_hi = c_hi + slack - W, w_lo = c_lo - slack - W1;
            if (w_hi > 0.0) {
                ew = fb_expo(w_hi);
                const bool draw = !(w_lo > 0.0);  // the walk may stop here
                rw = edge || draw || ew != fb_expo(w_lo);
                ex = ex || rw || !fb_alike(ql, qh, ew, dw);
                if (draw) {
                    atomicMin(&sh.first, static_cast<uint32_t>(b));
                    atomicMax(&sh.last, static_cast<uint32_t>(b));
                }
            }
            ++seen;
            n_elem += c;
            expo_end = static_cast<uint32_t>(fb_expo(A1 * (1.0 - kFbDrift)));
            if (ex) {
                n_items += c;
                ++n_seg;
                if (c > kFbSegMost && (rc || rw)) sh.bad = 1u;
                atomicOr(&sh.mask[b >> 5], 1u << (b & 31));
                sh.w[i] = static_cast<uint32_t>(ea) | (static_cast<uint32_t>(ew) << 8) | (rc ? kSegReplayCum : 0u) |
                          (rw ? kSegReplayWalk : 0u) | (ew ? kSegInWalk : 0u);
            } else {
                s_cum += static_cast<double>(c) * static_cast<double>(dc);
                s_walk += static_cast<double>(c) * static_cast<double>(dw);
                sh.w[i] = dc | (static_cast<uint32_t>(ew) << 24);
            }
        }
        at += c;
        W = W1;
    });
    uint32_t G, segs, elems;
    double cum_all, walk_all;
    double cum = s_cum, walk = s_walk;
    uint32_t off = n_items, seg = n_seg, elems_at = n_elem, unused = 0, none_all;
    fb_scan_3<kFW>(off, seg, cum, sh.sd, sh.su, sh.sv, G, segs, cum_all);
    fb_scan_3<kFW>(elems_at, unused, walk, sh.sd, sh.su, sh.sv, elems, none_all, walk_all);
    if (sh.bad || segs > static_cast<uint32_t>(kFbSegs)) {
        if (tid == 0) meta[kMetaStatus] = kStatusToSort;
        return;
    }
    const uint32_t draw0 = sh.first, draw1 = sh.last;
    at = before;
    if (seen != 0u) {
        uint32_t left = seen;
        each([&](int b, int i, uint32_t c) {
            if (left == 0u) return;
            --left;
            const uint32_t w = sh.w[i];
            if (static_cast<uint32_t>(b) == draw0) sh.off0 = off;
            if ((sh.mask[b >> 5] >> (b & 31)) & 1u) {
                r.bin[b] = off;
                r.seg[seg] = FbSeg{off, c, at, w, cum, walk, 0u, 0u};
                ++seg;
                off += c;
            } else {
                cum += static_cast<double>(c) * static_cast<double>(w & 0xffffffu);
                walk += static_cast<double>(c) * static_cast<double>(walk_ulps(b, static_cast<int>(w >> 24)));
            }
            if (static_cast<uint32_t>(b) == draw1) sh.off1 = off;
            at += c;
        });
        if (at == elems) r.seg[segs] = FbSeg{G, 0u, elems, expo_end | kSegReplayCum, cum_all, walk_all, 0u, 0u};  // the list's end
    }
    __syncthreads();
    for (int i = tid; i < kBins / 32; i += kFT) r.mask[i] = sh.mask[i];
    if (tid == 0) {
        const bool none = draw0 == 0xffffffffu;
        r.scal[kScShift] = shift;
        r.scal[kScInv] = f2u(inv);
        r.scal[kScDrawBin] = none ? 0u : draw0;
        r.scal[kScDrawItem] = sh.off0;
        r.scal[kScDrawEnd] = none ? 0u : sh.off1;
        r.scal[kScSegs] = segs;
        r.scal[kScLarge] = 0u;
        // whether the list ends where the reference's sums do: the row's end,
        // or the min-p cut
        r.scal[kScCut] = elems == static_cast<uint32_t>(V) || elems == sh.cut_elem ? 1u : 0u;
        meta[kMetaItems] = G;
        meta[kMetaStatus] = kStatusOk;
    }
}

// 4. The expanded bins' tokens to their items, in no order, and the sum of the
//    probabilities of the bins before the draw's. Streaming reads of the exps;
//    about one token in ten is expanded in near-uniform rows. Places are taken
//    from LDS counters: a part counts its tokens of each expanded bin first and
//    takes its share of the bin's items with one global atomic (the part is in
//    cache for its second read). With an atomic per token, 256 flat rows took
//    204 us and 64 peaked rows 27.
struct CollectShared {
    uint32_t next[kFbMaxBins];
    uint32_t mask[kFbMaxBins / 32];
    double sums[kFW];
};
__device__ __forceinline__ void fb_collect(const DevArgs& a, int row, int part, int parts, CollectShared& sh) {
    const int tid = threadIdx.x;
    ge_sample_params p;
    if (!fb_serves(a, row, p) || fb_meta(a, row)[kMetaStatus] != kStatusOk) return;
    const int bins = a.fo_bins;
    const FbRow r = fb_row(a, row, bins);
    for (int i = tid; i < bins / 32; i += kFT) sh.mask[i] = r.mask[i];
    for (int i = tid; i < bins; i += kFT) sh.next[i] = parts == 1 ? r.bin[i] : 0u;
    const uint32_t shift = r.scal[kScShift];
    const float inv = u2f(r.scal[kScInv]);
    const uint32_t draw = r.scal[kScDrawBin];
    __syncthreads();
    int lo, hi;
    fb_part(a, part, parts, lo, hi);
    const float* pes = fb_exp_array(a, row);
    uint64_t* items = a.fo_items + static_cast<int64_t>(row) * a.fo_items_stride;
    auto expanded = [&](uint32_t b) { return ((sh.mask[b >> 5] >> (b & 31u)) & 1u) != 0u; };
    if (parts > 1) {
        fb_stream<4>(pes, true, lo, hi, tid, [&](int, float x0, float x1, float x2, float x3, int n) {
            const float x[4] = {x0, x1, x2, x3};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t b = fb_bin(x[j], shift, static_cast<uint32_t>(bins));
                if (j < n && expanded(b)) atomicAdd(&sh.next[b], 1u);
            }
        });
        __syncthreads();
        for (int i = tid; i < bins; i += kFT) {
            const uint32_t c = sh.next[i];
            if (c) sh.next[i] = atomicAdd(&r.bin[i], c);
        }
        __syncthreads();
    }
    double sum = 0.0;
    fb_stream<4>(pes, true, lo, hi, tid, [&](int i, float x0, float x1, float x2, float x3, int n) {
        const float x[4] = {x0, x1, x2, x3};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (j < n) {
                const uint32_t b = fb_bin(x[j], shift, static_cast<uint32_t>(bins));
                if (b < draw) sum += static_cast<double>(x[j] * inv);
                if (expanded(b)) {
                    const uint32_t at = atomicAdd(&sh.next[b], 1u);
                    items[at] = (static_cast<uint64_t>(f2u(x[j])) << 32) | (0xffffffffu - static_cast<uint32_t>(i + j));
                }
            }
        }
    });
    sum = wave::sum_f64(sum);
    if ((tid & 63) == 0) sh.sums[tid >> 6] = sum;
    __syncthreads();
    if (tid == 0) {
        double t = 0.0;
        for (int w = 0; w < kFW; ++w) t += sh.sums[w];
        r.pbef[part] = t;
    }
}

// Each key's rank among a wave's n keys (kV per lane, key v of lane l the
// (64 v + l)-th; zero past n): how many are larger.
template <int kV>
__device__ __forceinline__ void fb_rank(const uint32_t (&key)[kV], uint32_t n, uint32_t (&rank)[kV]) {
#pragma unroll
    for (int v = 0; v < kV; ++v) rank[v] = 0;
#pragma unroll
    for (int w = 0; w < kV; ++w) {
        const int m = min(static_cast<int>(n) - 64 * w, 64);
#pragma unroll 1
        for (int c = 0; c < m; c += 8) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t k = wave::readlane(key[w], c + i);
#pragma unroll
                for (int v = 0; v < kV; ++v) rank[v] += k > key[v] ? 1u : 0u;
            }
        }
    }
}

// 5. Each expanded bin: the ulps its tokens add where it is not replayed (a
//    bin with a tie among them is replayed after all), and a replayed bin's
//    tokens by (exp descending, index ascending): one wave per bin by counting
//    the larger keys, the workgroup by a bitonic sort for the rare larger ones.
//    Bound by the counting. Exps of one bin differ in `shift` low bits only:
//    where these and the token's index fit 32 bits (near-uniform rows, whose
//    bins hold up to 120 tokens) the keys are ranked as 32-bit words from
//    registers; other bins rank 64-bit keys against an LDS broadcast.
//    256 near-uniform rows of V = 262,144: 98 us with 64-bit keys for all, 66 so;
//    16 workgroups a row measure the same, 5 (all resident at once) 79.
struct OrderShared {
    uint64_t stage[kFbSegMost];
};
template <int kThreads>
__device__ __forceinline__ void fb_order(const DevArgs& a, int row, int block, int blocks, OrderShared& sh) {
    constexpr int kWaves = kThreads / 64;
    constexpr int kMy = std::min(kFbWaveSeg, static_cast<int>(kFbSegMost) / kWaves) / 64;  // keys per lane
    constexpr uint32_t kWaveSeg = kMy * 64;
    const int tid = threadIdx.x, lane = __lane_id(), wave = tid >> 6;
    ge_sample_params p;
    if (!fb_serves(a, row, p) || fb_meta(a, row)[kMetaStatus] != kStatusOk) return;
    const FbRow r = fb_row(a, row, a.fo_bins);
    const int segs = static_cast<int>(r.scal[kScSegs]);
    const float inv = u2f(r.scal[kScInv]);
    const uint32_t shift = r.scal[kScShift], last_bin = static_cast<uint32_t>(a.fo_bins) - 1u;
    const int idx_bits = 32 - __clz(a.vocab - 1);
    const bool narrow = static_cast<int>(shift) + idx_bits <= 32;
    uint64_t* items = a.fo_items + static_cast<int64_t>(row) * a.fo_items_stride;
    uint64_t* mine = sh.stage + wave * kWaveSeg;
    bool large = false;
    // A wave reads 64 records at once (lane l: its l-th, the waves taking bins
    // in turn) and passes those with nothing to do, the single tokens of the
    // head above all; the next bin's first keys are in flight while one is
    // worked on.
    auto work = [&](uint32_t info, uint32_t n) {
        return n > 1u || !(info & kSegReplayCum) || ((info & kSegInWalk) && !(info & kSegReplayWalk));
    };
    const int turn = blocks * kWaves;
    for (int c0 = block * kWaves + wave; c0 < segs; c0 += turn * 64) {
      const int mine_s = c0 + lane * turn;
      const bool have = mine_s < segs;
      const uint32_t r_off = have ? r.seg[mine_s].item : 0u, r_n = have ? r.seg[mine_s].n : 0u;
      const uint32_t r_info = have ? r.seg[mine_s].info : 0u;
      uint64_t todo = __ballot(have && work(r_info, r_n));
      auto first_keys = [&](int l) {
          const uint32_t o = wave::readlane(r_off, l), m = wave::readlane(r_n, l);
          return items[o + min(static_cast<uint32_t>(lane), m - 1u)];
      };
      uint64_t next = todo ? first_keys(__builtin_ctzll(todo)) : 0ull;
      while (todo) {
        const int l = static_cast<int>(__builtin_ctzll(todo));
        todo &= todo - 1ull;
        const int s = c0 + l * turn;
        const uint32_t off = wave::readlane(r_off, l), n = wave::readlane(r_n, l);
        uint32_t info = wave::readlane(r_info, l);
        const bool sum_c = !(info & kSegReplayCum);
        const bool sum_w = (info & kSegInWalk) && !(info & kSegReplayWalk);
        const uint64_t key0 = static_cast<uint32_t>(lane) < n ? next : 0ull;
        if (todo) next = first_keys(__builtin_ctzll(todo));
        if (sum_c || sum_w) {
            const int uc = static_cast<int>(info & 0xffu) - 150, uw = static_cast<int>((info >> 8) & 0xffu) - 150;
            uint32_t tc = 0, tw = 0;
            bool oc = false, ow = false;  // a tie, an addend past the binade, or a sum past it
            for (uint32_t i = static_cast<uint32_t>(lane); i < n; i += 64u) {
                const uint64_t key = i < 64u ? key0 : items[off + i];
                const uint32_t qb = f2u(u2f(static_cast<uint32_t>(key >> 32)) * inv);
                uint32_t D;
                bool tie, big;
                chain::step_bits(qb, uc, D, tie, big);
                tc += min(D, 0x1000000u);
                oc = oc || tie || big || tc > 0x1000000u;
                tc = min(tc, 0x1000000u);
                chain::step_bits(qb, uw, D, tie, big);
                tw += min(D, 0x1000000u);
                ow = ow || tie || big || tw > 0x1000000u;
                tw = min(tw, 0x1000000u);
            }
            // (a lane's sum stays below 2^25, so the wave's fits 31 bits)
            if (sum_c && __ballot(oc)) info |= kSegReplayCum;
            if (sum_w && __ballot(ow)) info |= kSegReplayWalk;
            const uint32_t dc = wave::incl_add(tc), dw = wave::incl_add(tw);
            if (lane == 63) {
                r.seg[s].info = info;
                r.seg[s].scum = dc;
                r.seg[s].swalk = dw;
            }
        }
        if (!(info & (kSegReplayCum | kSegReplayWalk))) continue;
        // (the last bin holds every smaller exp too)
        const bool words = narrow && n <= 256u &&
                           wave::readlane(fb_bin(u2f(static_cast<uint32_t>(key0 >> 32)), shift, last_bin + 1u), 0) != last_bin;
        auto by_words = [&](auto kv) {
            constexpr int kV = decltype(kv)::value;
            uint64_t key[kV];
            uint32_t word[kV], rank[kV];
#pragma unroll
            for (int v = 0; v < kV; ++v) {
                const uint32_t i = static_cast<uint32_t>(v) * 64u + static_cast<uint32_t>(lane);
                key[v] = v == 0 ? key0 : items[off + min(i, n - 1u)];
            }
            // ((2^shift - 1 - the exp's distance into the bin), then the index's complement)
            const uint32_t below = (1u << shift) - 1u, idx_mask = (1u << idx_bits) - 1u;
#pragma unroll
            for (int v = 0; v < kV; ++v) {
                const uint32_t hi = below - ((kOne - static_cast<uint32_t>(key[v] >> 32)) & below);
                const bool in = static_cast<uint32_t>(v) * 64u + static_cast<uint32_t>(lane) < n;
                word[v] = in ? (hi << idx_bits) | (static_cast<uint32_t>(key[v]) & idx_mask) : 0u;
            }
            fb_rank<kV>(word, n, rank);
#pragma unroll
            for (int v = 0; v < kV; ++v)
                if (static_cast<uint32_t>(v) * 64u + static_cast<uint32_t>(lane) < n) items[off + rank[v]] = key[v];
        };
        if (words) {
            if (n <= 64u) by_words(std::integral_constant<int, 1>{});
            else if (n <= 128u) by_words(std::integral_constant<int, 2>{});
            else by_words(std::integral_constant<int, 4>{});
        } else if (n <= 64u) {
            uint32_t rank = 0;
            for (uint32_t j = 0; j < n; ++j) rank += wave::readlane64(key0, static_cast<int>(j)) > key0 ? 1u : 0u;
            if (static_cast<uint32_t>(lane) < n) items[off + rank] = key0;
        } else if (n <= kWaveSeg) {
            uint64_t key[kMy];
            uint32_t rank[kMy];
#pragma unroll
            for (int v = 0; v < kMy; ++v) {
                const uint32_t i = static_cast<uint32_t>(v) * 64u + static_cast<uint32_t>(lane);
                key[v] = i < n ? items[off + i] : 0ull;
                rank[v] = 0;
                mine[i] = key[v];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            for (uint32_t j = 0; j < n; ++j) {
                const uint64_t k = mine[j];
#pragma unroll
                for (int v = 0; v < kMy; ++v)
                    if (static_cast<uint32_t>(v) * 64u < n) rank[v] += k > key[v] ? 1u : 0u;
            }
#pragma unroll
            for (int v = 0; v < kMy; ++v)
                if (static_cast<uint32_t>(v) * 64u + static_cast<uint32_t>(lane) < n) items[off + rank[v]] = key[v];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        } else {
            large = true;
            // (not the status word: other waves and workgroups of this kernel still
            // read that, and must all go on to the barriers below)
            if (n > kFbSegMost && lane == 0) r.scal[kScLarge] = 1u;
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(0);  // the flags written above are read below by every wave
    if (__syncthreads_or(large ? 1 : 0) == 0) return;
    for (int s0 = block * kWaves; s0 < segs; s0 += turn) {
        for (int s = s0; s < min(s0 + kWaves, segs); ++s) {
            const uint32_t off = r.seg[s].item, n = r.seg[s].n;
            // (block-uniform; the flags as this workgroup's waves left them)
            const uint32_t info = ld_l2(&r.seg[s].info);
            if (n <= kWaveSeg || n > kFbSegMost || !(info & (kSegReplayCum | kSegReplayWalk))) continue;
            uint32_t n2 = 1;
            while (n2 < n) n2 <<= 1;
            __syncthreads();
            for (uint32_t i = tid; i < n2; i += kThreads) sh.stage[i] = i < n ? items[off + i] : 0ull;
            for (uint32_t size = 2; size <= n2; size <<= 1) {
                for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
                    __syncthreads();
                    for (uint32_t q = tid; q < n2 / 2; q += kThreads) {
                        const uint32_t i = 2u * q - (q & (stride - 1u));
                        const uint64_t x = sh.stage[i], y = sh.stage[i + stride];
                        const bool desc = (i & size) == 0u;
                        if (desc ? x < y : x > y) {
                            sh.stage[i] = y;
                            sh.stage[i + stride] = x;
                        }
                    }
                }
            }
            __syncthreads();
            for (uint32_t i = tid; i < n; i += kThreads) items[off + i] = sh.stage[i];
        }
    }
}

// 6. The chains (generation.cpp:103-126): the replayed bins' probabilities in
//    LDS lists, one for the cumulative and one for the walk, cut into regions
//    of consecutive elements; the ulps of the bins between two regions are
//    added at once. One wave takes the lists 64 elements a step. Then the
//    near-boundary flag and the token. Latency-bound: about 150 steps of
//    dependent work per chain for near-uniform rows.
constexpr int kDrawList = 14336;    // replayed elements of one chain
constexpr int kDrawRegions = 512;   // their regions
constexpr int kDrawTies = 4096;     // tokens of one exp (kFbSegMost)

struct DrawList {
    union {
        uint32_t q[kDrawList];      // the probabilities' bits
        uint64_t tie[kDrawTies];    // (once the chains are done)
    };
    double before[kDrawRegions + 1];   // ulps of the bins before the region, from the row's start
    uint32_t pos[kDrawRegions + 1];    // its first list position; [n]: the list's length
    uint32_t item[kDrawRegions + 1];
    uint32_t elem[kDrawRegions + 1];
    uint32_t expo[kDrawRegions + 1];   // the accumulator's binade before it (0: no bins lie between, or none that add)
    int n;                             // regions
};
static_assert(kDrawList * 4 >= kDrawTies * 8, "the union");
struct DrawShared {
    DrawList list[2];  // cumulative, walk
    double sd[32];
    uint32_t su[32], sr[32];
    double s;
    uint32_t keep, pos, item, near_u, ok;
    int32_t token;
};

// Both chains' lists from the row's expanded bins: thread t takes consecutive
// records, and one workgroup scan places its regions and elements. False
// (block-uniform) when they do not fit.
template <int kThreads>
__device__ __forceinline__ bool draw_lists(const FbRow& r, int segs, const uint64_t* items, float inv, DrawShared& sh) {
    constexpr int kWaves = kThreads / 64;
    constexpr int kBatch = 4;  // records in flight
    constexpr uint32_t kReplay[2] = {kSegReplayCum, kSegReplayWalk};
    const int tid = threadIdx.x, wave = tid >> 6;
    const int count = segs + 1;  // with the list's end
    const int per = (count + kThreads - 1) / kThreads;
    const int s0 = min(tid * per, count), s1 = min(s0 + per, count);
    // f(record, chain, replayed, begins a region, follows the replayed tokens before it)
    auto each = [&](auto&& f) {
        const FbSeg p = r.seg[max(s0 - 1, 0)];
        bool prev[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) prev[x] = s0 > 0 && (p.info & kReplay[x]) != 0u;
        uint32_t next = p.elem + p.n;
        for (int b = s0; b < s1; b += kBatch) {
            FbSeg g[kBatch];
#pragma unroll
            for (int v = 0; v < kBatch; ++v) g[v] = r.seg[min(b + v, count - 1)];  // clamped: no conditional load
#pragma unroll
            for (int v = 0; v < kBatch; ++v) {
                if (b + v >= s1) continue;
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    const bool rep = (g[v].info & kReplay[x]) != 0u;
                    const bool follows = prev[x] && next == g[v].elem;  // no bins between
                    f(g[v], x, rep, rep && !(follows && g[v].n != 0u), follows);
                    prev[x] = rep;
                }
                next = g[v].elem + g[v].n;
            }
        }
    };
    double t[2] = {0.0, 0.0};  // the ulps of the expanded bins that are not replayed
    uint32_t n[2] = {0, 0}, at[2] = {0, 0};
    each([&](const FbSeg& g, int x, bool rep, bool start, bool) {
        if (rep) n[x] += g.n;
        else t[x] += static_cast<double>(x ? g.swalk : g.scum);
        at[x] += start ? 1u : 0u;
    });
    uint32_t n_all[2], r_all[2];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        const double ti = wave::incl_f64(t[x]);
        const uint32_t ni = wave::incl_add(n[x]), ri = wave::incl_add(at[x]);
        if ((tid & 63) == 63) {
            sh.sd[16 * x + wave] = ti;
            sh.su[16 * x + wave] = ni;
            sh.sr[16 * x + wave] = ri;
        }
        t[x] = ti - t[x];
        n[x] = ni - n[x];
        at[x] = ri - at[x];
    }
    static_assert(kWaves <= 16, "the scan's words");
    __syncthreads();
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        n_all[x] = r_all[x] = 0;
        for (int w = 0; w < kWaves; ++w) {
            if (w < wave) {
                t[x] += sh.sd[16 * x + w];
                n[x] += sh.su[16 * x + w];
                at[x] += sh.sr[16 * x + w];
            }
            n_all[x] += sh.su[16 * x + w];
            r_all[x] += sh.sr[16 * x + w];
        }
    }
    if (max(n_all[0], n_all[1]) > static_cast<uint32_t>(kDrawList) || max(r_all[0], r_all[1]) > static_cast<uint32_t>(kDrawRegions))
        return false;
    each([&](const FbSeg& g, int x, bool rep, bool start, bool follows) {
        DrawList& l = sh.list[x];
        if (start) {
            l.before[at[x]] = t[x] + (x ? g.walk : g.cum);
            l.pos[at[x]] = n[x];
            l.item[at[x]] = g.item;
            l.elem[at[x]] = g.elem;
            l.expo[at[x]] = follows ? 0u : x ? (g.info >> 8) & 0xffu : g.info & 0xffu;
            ++at[x];
        }
        if (rep) n[x] += g.n;
        else t[x] += static_cast<double>(x ? g.swalk : g.scum);
    });
    if (tid < 2) {
        sh.list[tid].n = static_cast<int>(r_all[tid]);
        sh.list[tid].pos[r_all[tid]] = n_all[tid];
    }
    __syncthreads();
    for (uint32_t i = tid; i < n_all[0] + n_all[1]; i += kThreads) {
        const int x = i < n_all[0] ? 0 : 1;
        const uint32_t k = x ? i - n_all[0] : i;
        DrawList& l = sh.list[x];
        uint32_t lo = 0, hi = r_all[x];  // the region: pos[lo] <= k < pos[lo + 1]
        while (hi - lo > 1u) {
            const uint32_t m = (lo + hi) >> 1;
            if (l.pos[m] <= k) lo = m;
            else hi = m;
        }
        l.q[k] = f2u(u2f(static_cast<uint32_t>(items[l.item[lo] + (k - l.pos[lo])] >> 32)) * inv);
    }
    __syncthreads();
    return true;
}

// One wave takes list elements [k, limit) from the accumulator s (asc: s +=
// q, until s >= thr; desc: s -= q, until s <= q). Returns 1 at a stop (k: its
// position), 0 at the limit, -1 where the bins between two regions do not fit
// the binade the plan took them in.
template <bool kDesc>
__device__ __forceinline__ int draw_chain(const DrawList& l, uint32_t& k, uint32_t limit, int& region, float& s, float thr) {
    const int lane = __lane_id();
    const uint32_t n_all = l.pos[l.n];
    uint32_t rend = l.pos[region + 1];
    // (the cumulative ends where a region begins: the bins before it count too)
    while (k < limit || (!kDesc && k == rend && region + 1 < l.n)) {
        const chain::StepBits b = chain::binade_bits(f2u(s));
        const uint32_t tm = kDesc ? 0u : chain::threshold_bits(f2u(thr), b.uexp);
        if (k == rend) {  // the bins between this region and the next
            if (region + 1 >= l.n) return -1;
            // The plan took them in one binade. In a higher one their ulps are
            // others, unless they add nothing: then they add nothing there
            // either. In a lower one they may add even where the plan's add
            // nothing.
            const double jump = l.before[region + 1] - l.before[region];
            const uint32_t planned = l.expo[region + 1], have = static_cast<uint32_t>(b.uexp + 150);
            if (planned != 0u) {
                const double m = static_cast<double>(b.m);
                if (have < planned || (have > planned && jump != 0.0)) return -1;
                if (kDesc ? m - jump < static_cast<double>(b.lo)
                          : (m + jump > static_cast<double>(chain::kHiF) || m + jump >= static_cast<double>(tm)))
                    return -1;
                s = u2f(chain::rebuild_bits(f2u(s), static_cast<uint32_t>(kDesc ? m - jump : m + jump)));
            }
            ++region;
            rend = l.pos[region + 1];
            continue;
        }
        const uint32_t end = min(rend, limit);
        const bool on = k + static_cast<uint32_t>(lane) < end;
        const uint32_t qb = l.q[min(k + static_cast<uint32_t>(lane), n_all - 1u)];
        uint32_t D;
        bool tie, big;
        chain::step_bits(qb, b.uexp, D, tie, big);
        D = on ? D : 0u;
        const uint32_t incl = wave::incl_add(D);  // at most 64 * 2^24
        const bool out = kDesc ? b.m < b.lo + incl : (b.m + incl > chain::kHiF || b.m + incl >= tm);
        const uint64_t ev = __ballot(on && (out || tie || big));
        if (ev == 0ull) {
            const uint32_t t = wave::readlane(incl, 63);
            s = u2f(chain::rebuild_bits(f2u(s), kDesc ? b.m - t : b.m + t));
            k = min(k + 64u, end);
            continue;
        }
        const int f = static_cast<int>(__builtin_ctzll(ev));
        const uint32_t t = wave::readlane(incl, f) - wave::readlane(D, f);
        const float q = u2f(wave::readlane(qb, f));
        s = u2f(chain::rebuild_bits(f2u(s), kDesc ? b.m - t : b.m + t));
        k += static_cast<uint32_t>(f);
        if (kDesc) {
            if (s <= q) return 1;
            s = s - q;
        } else {
            s = s + q;
            if (s >= thr) return 1;
        }
        ++k;
    }
    return 0;
}

template <int kThreads>
__device__ __forceinline__ void fb_draw(const DevArgs& a, int row, int parts, DrawShared& sh) {
    constexpr int kWaves = kThreads / 64;
    const int tid = threadIdx.x, lane = __lane_id(), wave = tid >> 6;
    const ge_sample_params p = a.row_params ? a.row_params[row] : a.params;
    uint32_t k;
    if (!full_order_row(p, a.vocab, k)) return;
    if (row_done(a, row)) {
        if (tid == 0) skipped_row(a, row);
        return;
    }
    uint32_t* meta = fb_meta(a, row);
    if (meta[kMetaStatus] != kStatusOk) return;  // the sort-based pass serves the row
    const int V = a.vocab;
    const FbRow r = fb_row(a, row, a.fo_bins);
    const int segs = static_cast<int>(r.scal[kScSegs]);
    const uint64_t* items = a.fo_items + static_cast<int64_t>(row) * a.fo_items_stride;
    const float inv = u2f(r.scal[kScInv]);
    const int draw0 = static_cast<int>(r.scal[kScDrawItem]), draw1 = static_cast<int>(r.scal[kScDrawEnd]);
    const bool whole = r.scal[kScCut] != 0u;
    bool ok = r.scal[kScLarge] == 0u && draw_lists<kThreads>(r, segs, items, inv, sh);
    const float u = a.uniforms[row];
    float choice = 0.0f;
    if (ok && wave == 0) {
        const DrawList& lc = sh.list[0];
        const DrawList& lw = sh.list[1];
        const uint32_t n_all = lc.pos[lc.n];
        const float q0 = u2f(lc.q[0]);
        const float minimum = q0 * p.min_p;
        bool good = lc.n > 0 && lc.elem[0] == 0u && n_all > 0u;
        // generation.cpp:106-108: the first element e >= 1 with p_e < minimum
        // (the list holds the whole bin that has it).
        uint32_t limit = n_all;
        if (q0 < minimum) limit = 1u;
        else if (minimum > 0.0f) limit = wave_partition_point(1u, n_all, [&](uint32_t i) { return !(u2f(lc.q[i]) < minimum); });
        uint32_t kc = 1u;
        int rc = 0;
        float s = q0;
        uint32_t keep = 1u;
        if (good && !(q0 < minimum) && q0 >= p.top_p && lc.n > 1 && lc.pos[1] == 1u && lc.elem[1] > 1u) {
            keep = 2u;  // the first check comes after the second element, which adds nothing
        } else if (good && !(q0 < minimum)) {
            const int hit = draw_chain<false>(lc, kc, limit, rc, s, p.top_p);
            if (hit < 0) good = false;
            else if (hit == 1) keep = lc.elem[rc] + (kc - lc.pos[rc]) + 1u;
            else if (limit < n_all || whole) keep = lc.elem[rc] + (kc - lc.pos[rc]);
            else good = false;  // the list ends before the sums do
        }
        // random.h:1864-1871 and generation.cpp:118-124.
        choice = u * (s - 0.0f) + 0.0f;
        uint32_t pos = 0u, item = lc.item[0];
        if (good && choice > 0.0f && choice < __builtin_inff()) {
            good = lw.n > 0 && lw.elem[0] == 0u;
            if (good) {
                // the list's elements before `keep`
                const uint32_t lr = wave_partition_point(0u, static_cast<uint32_t>(lw.n), [&](uint32_t i) { return lw.elem[i] < keep; }) - 1u;
                const uint32_t wlim = lw.pos[lr] + min(lw.pos[lr + 1u] - lw.pos[lr], keep - lw.elem[lr]);
                uint32_t kw = 0u;
                int rw = 0;
                float c = choice;
                const int hit = draw_chain<true>(lw, kw, wlim, rw, c, 0.0f);
                if (hit == 0) {  // the walk passes every kept element: the last one
                    good = kw > 0u && lw.elem[rw] + (kw - lw.pos[rw]) == keep;
                    --kw;
                }
                good = good && hit >= 0;
                pos = lw.elem[rw] + (kw - lw.pos[rw]);
                item = lw.item[rw] + (kw - lw.pos[rw]);
            }
        } else if (!(choice <= 0.0f)) {
            good = false;
        }
        if (lane == 0) {
            sh.ok = good ? 1u : 0u;
            sh.keep = keep;
            sh.pos = pos;
            sh.item = item;
            sh.s = static_cast<double>(choice);
            sh.token = -1;
        }
    }
    __syncthreads();
    ok = ok && sh.ok != 0u;
    const uint32_t pos = sh.pos, keep = sh.keep;
    const int item = static_cast<int>(sh.item);
    bool near = false;
    if (ok) {
        // Near-boundary flag: double sums of the probabilities before and
        // through the chosen position; the sum before the draw's bins is
        // fb_collect's, the rest its single tokens.
        const double ch = sh.s;
        double before = 0.0;
        bool nb = false, na = false;
        if (pos > 0u) {
            // (item == pos: every token before it is in the list, whatever the
            // plan expected: a draw one token before its range sent 3 peaked rows in
            // 15,000 to the sort)
            const bool head = static_cast<uint32_t>(item) == pos;
            if (!head && (item < draw0 || item >= draw1)) {
                ok = false;
            } else {
                double t = 0.0;
                for (int i = (head ? 0 : draw0) + tid; i < item; i += kThreads)
                    t += static_cast<double>(u2f(static_cast<uint32_t>(items[i] >> 32)) * inv);
                t = wave::sum_f64(t);
                if (lane == 0) sh.sd[wave] = t;
                __syncthreads();
                before = head ? 0.0 : wave::sum_f64(lane < parts ? r.pbef[lane] : 0.0);
                for (int v = 0; v < kWaves; ++v) before += sh.sd[v];
                ok = near_decided(ch, before, near_sum_error(pos), nb);
            }
        }
        const float q = u2f(static_cast<uint32_t>(items[item] >> 32)) * inv;
        ok = ok && near_decided(ch, before + static_cast<double>(q), near_sum_error(pos), na);
        near = (pos > 0u && nb) || (pos + 1u < keep && na);
    }
    if (!ok) {  // block-uniform
        if (tid == 0) meta[kMetaStatus] = kStatusToSort;
        return;
    }
    // 7. The token: among the tokens of the chosen exp (neighbours in the list),
    //    the one of its rank by (final value descending, index ascending).
    const int32_t* hist;
    int H;
    history_of(a, row, hist, H);
    const bool pen = H > 0 && !(p.repetition_penalty == 1.0f);
    uint32_t* bitmap = a.fo_bitmap + static_cast<int64_t>(row) * a.fo_bitmap_words;
    const float* rowp = static_cast<const float*>(a.logits) + static_cast<int64_t>(row) * a.row_stride;
    const uint32_t peb = static_cast<uint32_t>(items[item] >> 32);
    const int G = static_cast<int>(meta[kMetaItems]);
    // (the tokens of one exp lie in one bin; bins beside it hold other exps)
    auto same = [&](int i) { return i >= 0 && i < G && static_cast<uint32_t>(items[i] >> 32) == peb; };
    int is = item, ie = item;  // (every wave finds the same run)
    for (;;) {
        const uint64_t m = __ballot(same(is - 1 - lane));
        const int n = m == ~0ull ? 64 : static_cast<int>(__builtin_ctzll(~m));
        is -= n;
        if (n < 64) break;
    }
    for (;;) {
        const uint64_t m = __ballot(same(ie + 1 + lane));
        const int n = m == ~0ull ? 64 : static_cast<int>(__builtin_ctzll(~m));
        ie += n;
        if (n < 64) break;
    }
    const int n_tie = ie - is + 1;
    uint64_t* tie = sh.list[0].tie;
    if (n_tie == 1) {
        if (tid == 0) sh.token = static_cast<int32_t>(composite_index(items[item]));
    } else {  // (at most kFbSegMost: one exp lies in one bin)
        for (int i = tid; i < n_tie; i += kThreads) {
            const uint32_t idx = composite_index(items[is + i]);
            float v = softcap(rowp[idx], p.softcap);
            if (pen && ((bitmap[idx >> 5] >> (idx & 31u)) & 1u)) v = penalize(v, p.repetition_penalty);
            tie[i] = composite(order_key(v), idx);
        }
        __syncthreads();
        const uint32_t want = static_cast<uint32_t>(item - is);
        for (int i = tid; i < n_tie; i += kThreads) {
            const uint64_t x = tie[i];
            uint32_t rank = 0;
            for (int j = 0; j < n_tie; ++j) rank += tie[j] > x ? 1u : 0u;
            if (rank == want) sh.token = static_cast<int32_t>(composite_index(x));
        }
    }
    __syncthreads();
    // The bitmap is all zero again after every call (cleared from the history
    // before the token is appended: a full ring's history is the ring).
    if (pen) {
        for (int i = tid; i < H; i += kThreads) {
            const int32_t id = hist[i];
            if (id >= 0 && id < V) bitmap[id >> 5] = 0u;
        }
        __syncthreads();
    }
    if (tid == 0) emit_row(a, row, sh.token, u2f(peb) * inv, near ? GE_FLAG_NEAR_BOUNDARY : 0);
}

// ---- launches ----------------------------------------------------------------

constexpr int kOT = 256;  // threads of fb_order_kernel
constexpr int kDT = 512;  // and of fb_draw_kernel

__global__ __launch_bounds__(kFT) void fb_range_kernel(DevArgs a) {
    __shared__ RangeShared sh;
    fb_range(a, blockIdx.y, blockIdx.x, gridDim.x, sh);
}
__global__ __launch_bounds__(kFT) void fb_exps_kernel(DevArgs a) {
    __shared__ ExpsShared sh;
    fb_exps(a, blockIdx.y, blockIdx.x, gridDim.x, sh);
    if (blockIdx.x == 0 && threadIdx.x == 0) fb_clear_left(a, blockIdx.y);
}
template <int kPer>
__global__ __launch_bounds__(kFT) void fb_plan_kernel(DevArgs a, int parts) {
    __shared__ PlanShared sh;
    fb_plan<kPer>(a, blockIdx.x, parts, sh);
}
__global__ __launch_bounds__(kFT) void fb_collect_kernel(DevArgs a) {
    __shared__ CollectShared sh;
    fb_collect(a, blockIdx.y, blockIdx.x, gridDim.x, sh);
}
__global__ __launch_bounds__(kOT) void fb_order_kernel(DevArgs a) {
    __shared__ OrderShared sh;
    fb_order<kOT>(a, blockIdx.y, blockIdx.x, gridDim.x, sh);
}
__global__ __launch_bounds__(kDT) void fb_draw_kernel(DevArgs a, int parts) {
    __shared__ DrawShared sh;
    fb_draw<kDT>(a, blockIdx.x, parts, sh);
}

// Calls with per-row parameters: one workgroup takes a row through every stage.
// The host cannot tell whether any row needs this path, and six launches cost
// 20 us when none does; a served row takes longer than spread over the chip (its
// exps run on one CU), but many rows run side by side.
union RowShared {
    RangeShared range;
    ExpsShared exps;
    PlanShared plan;
    CollectShared collect;
    OrderShared order;
    DrawShared draw;
    __device__ RowShared() {}
};
// The stage's stores and atomics done and seen by the workgroup's loads (some
// were made in L2, past the CU's L1).
__device__ __forceinline__ void stage_done() {
    __threadfence();
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
}
template <int kPer>
__global__ __launch_bounds__(kFT) void fb_row_kernel(DevArgs a) {
    __shared__ RowShared sh;
    const int row = blockIdx.x;
    ge_sample_params p;
    uint32_t k;
    if (threadIdx.x == 0) fb_clear_left(a, row);
    fb_range(a, row, 0, 1, sh.range);
    if (!fb_serves(a, row, p)) {  // (block-uniform) done rows are reported by the draw
        if (full_order_row(p, a.vocab, k) && row_done(a, row)) fb_draw<kFT>(a, row, 1, sh.draw);
        return;
    }
    stage_done();
    fb_exps(a, row, 0, 1, sh.exps);
    stage_done();
    fb_plan<kPer>(a, row, 1, sh.plan);
    stage_done();
    fb_collect(a, row, 0, 1, sh.collect);
    stage_done();
    fb_order<kFT>(a, row, 0, 1, sh.order);
    stage_done();
    fb_draw<kFT>(a, row, 1, sh.draw);
}

}  // namespace

hipError_t launch_binned(const DevArgs& args, hipStream_t stream) {
    DevArgs a = args;
    a.fo_bins = fb_bins(a.vocab, a.rows);
    // Parts per row: about two workgroups per CU in all, at most one per step.
    // (Against 256 and 1,024 in all, near-uniform rows of V = 262,144: 32 rows 223,
    // 216, 248 us, 64 264, 259, 274, 96 351, 373, 351, 256 532, 522, 544; of V = 50,257:
    // 64 161, 153, 171, 96 187, 186, 197, 256 250, 241, 266. 256 loses only at 96.)
    const int steps = (a.vocab + kFStep - 1) / kFStep;
    const int parts = std::max(1, std::min({steps, kFbParts, (512 + a.rows - 1) / a.rows}));
    const dim3 grid(static_cast<unsigned>(parts), static_cast<unsigned>(a.rows));
    const int bins = a.fo_bins;
    if (a.row_params) {
        const dim3 all(static_cast<unsigned>(a.rows));
        switch (bins / kFT) {
            case 2: hipLaunchKernelGGL(fb_row_kernel<2>, all, dim3(kFT), 0, stream, a); break;
            case 4: hipLaunchKernelGGL(fb_row_kernel<4>, all, dim3(kFT), 0, stream, a); break;
            case 8: hipLaunchKernelGGL(fb_row_kernel<8>, all, dim3(kFT), 0, stream, a); break;
            default: hipLaunchKernelGGL(fb_row_kernel<16>, all, dim3(kFT), 0, stream, a); break;
        }
        return hipGetLastError();
    }
    hipLaunchKernelGGL(fb_range_kernel, grid, dim3(kFT), 0, stream, a);
    hipLaunchKernelGGL(fb_exps_kernel, grid, dim3(kFT), 0, stream, a);
    const dim3 rows(static_cast<unsigned>(a.rows));
    switch (bins / kFT) {
        case 2: hipLaunchKernelGGL(fb_plan_kernel<2>, rows, dim3(kFT), 0, stream, a, parts); break;
        case 4: hipLaunchKernelGGL(fb_plan_kernel<4>, rows, dim3(kFT), 0, stream, a, parts); break;
        case 8: hipLaunchKernelGGL(fb_plan_kernel<8>, rows, dim3(kFT), 0, stream, a, parts); break;
        default: hipLaunchKernelGGL(fb_plan_kernel<16>, rows, dim3(kFT), 0, stream, a, parts); break;
    }
    // One part for many rows: its places need no counting pass. Whole calls with
    // the rule, with one part always and with all parts always, near-uniform
    // rows of V = 262,144: 64 rows 263, 283, 264 us, 96 352, 356, 353, 128 363, 364,
    // 353, 192 491, 492, 513, 256 535, 534, 579; V = 50,257: 64 161, 165, 161, 96 188,
    // 184, 188, 128 all 199, 256 250, 250, 262.
    const int cparts = a.rows >= 128 ? 1 : parts;
    hipLaunchKernelGGL(fb_collect_kernel, dim3(static_cast<unsigned>(cparts), static_cast<unsigned>(a.rows)), dim3(kFT), 0,
                       stream, a);
    // (half or twice as many workgroups: within 2% at 1 to 256 rows)
    const unsigned ob = static_cast<unsigned>(std::max(4, std::min(128, 2048 / a.rows)));
    hipLaunchKernelGGL(fb_order_kernel, dim3(ob, static_cast<unsigned>(a.rows)), dim3(kOT), 0, stream, a);
    hipLaunchKernelGGL(fb_draw_kernel, rows, dim3(kDT), 0, stream, a, cparts);
    return hipGetLastError();
}

}  // namespace ge
