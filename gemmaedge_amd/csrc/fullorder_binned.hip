// Full-order sampling of f32 rows without a sort (top-k disabled: k = V,
// src/generation.cpp:80).
//
// The reference sorts the row and then adds the probabilities one by one in
// float: the top-p cumulative, and the draw's subtract walk. Inside one
// binade of the accumulator such a sum moves by whole ulps, and the number of
// ulps that an addend q adds, round(q / ulp), does not depend on the order
// (chain_math.h; an exact tie does, through the accumulator's parity). So the
// order only matters where the accumulator changes binade, where an addend ties,
// and where the sum stops. Everywhere else a run of neighbouring addends that
// all round to the same number of ulps is one item (count, any of the
// addends) of the closed-form chain. A row of V = 262,144 near-uniform
// logits then has some 25,000 items in place of 262,144 sorted tokens, and a
// confident row a few thousand.
//
//   fb_range    marks the history ids; the row's largest final value and
//               smallest raw one
//   fb_exps     every token's exp((v - max) / T), kept; their sum; their
//               histogram in bins of equal width in the float's bits
//   fb_plan     1 / denominator; per bin the probabilities' sum before it and
//               the walk's, following the float sums' rounding; which bins
//               must be expanded into single tokens (a binade change, the
//               top-p, min-p or draw stop, or not all addends alike there)
//   fb_collect  the expanded bins' tokens; the sum of the probabilities
//               before the bins the draw can end in
//   fb_order    the expanded bins' tokens in order
//   fb_draw     the chains over the items, the token, and a check that every
//               unexpanded bin was passed in the binade the plan assumed
//
// Results are exact for any plan: fb_draw checks what the plan assumed
// and otherwise leaves the row to the sort-based pass, as do rows that this
// path does not serve (NaN or infinite maxima, a denominator whose
// reciprocal the sum's error interval leaves open, expanded bins of more than
// kFbSegMost tokens).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>

#include "chain_block.h"
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
constexpr uint32_t kLeast = 0x2f800000u;  // 2^-32: smaller exps share the last bin at most
constexpr uint32_t kFbHead = 1024;     // tokens always expanded
constexpr int kFbWaveSeg = 512;        // tokens of a bin that one wave orders
constexpr uint32_t kFbSegMost = 4096;  // tokens of an expanded bin at most
constexpr double kFbDrift = 0x1p-11;   // the plan's relative margin on a float sum
constexpr uint64_t kFbRegular = 1ull << 63;  // an item that stands for a whole bin

// The row's area in fo_tiles.
struct FbRow {
    uint32_t* bin;    // [bins] counts, then the expanded bins' next item
    uint32_t* pmax;   // [kFbParts] largest final key
    uint32_t* pmin;   // [kFbParts] smallest raw key
    double* psum;     // [kFbParts] sums of exps
    double* pbef;     // [kFbParts] sums of the probabilities before the draw's bins
    uint32_t* scal;   // [kScalWords]
    uint32_t* mask;   // [bins / 32] expanded bins
    uint32_t* seg;    // [3 * kFbSegs] item, tokens and first element of each expanded bin
};
enum : int { kScShift = 0, kScInv, kScDrawBin, kScDrawItem, kScDrawEnd, kScSegs, kScalWords = 64 };

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
    r.seg = r.mask + kFbMaxBins / 32;
    return r;
}
// The row's exps, in the upper half of its items (fb_half() items are left).
__device__ __forceinline__ int64_t fb_half(const DevArgs& a) { return a.fo_items_stride / 2; }
__device__ __forceinline__ float* fb_exp_array(const DevArgs& a, int row) {
    return reinterpret_cast<float*>(a.fo_items + static_cast<int64_t>(row) * a.fo_items_stride + fb_half(a));
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
__global__ __launch_bounds__(kFT) void fb_range_kernel(DevArgs a) {
    __shared__ uint32_t s[kFW];
    const int row = blockIdx.y, part = blockIdx.x, parts = gridDim.x, tid = threadIdx.x;
    ge_sample_params p;
    const int bins = fb_bins(a.vocab);
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
// from 1 down to the smallest one (2^-32 at least), over all bins.
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
__global__ __launch_bounds__(kFT) void fb_exps_kernel(DevArgs a) {
    __shared__ uint32_t hist_s[kFbMaxBins];
    __shared__ uint64_t tab[32];
    __shared__ double sums[kFW];
    __shared__ float s_vmax;
    __shared__ uint32_t s_shift;
    const int row = blockIdx.y, part = blockIdx.x, parts = gridDim.x, tid = threadIdx.x;
    ge_sample_params p;
    if (!fb_serves(a, row, p)) return;
    const int bins = fb_bins(a.vocab);
    const FbRow r = fb_row(a, row, bins);
    if (tid < 64) {
        float vm;
        uint32_t sh;
        fb_bin_shape(r, parts, bins, p, vm, sh);
        if (tid == 0) {
            s_vmax = vm;
            s_shift = sh;
        }
        if (tid < 32) tab[tid] = exp2_table(static_cast<uint32_t>(tid));
    }
    for (int i = tid; i < bins; i += kFT) hist_s[i] = 0u;
    __syncthreads();
    const float vmax = s_vmax;
    const uint32_t shift = s_shift;
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
    double sum = 0.0;
    fb_stream<4>(rowp, a.vec_ok != 0, lo, hi, tid, [&](int i, float x0, float x1, float x2, float x3, int n) {
        const uint32_t bits = pen && n ? bitmap[i >> 5] >> (i & 31) : 0u;
        const float x[4] = {x0, x1, x2, x3};
        float pe[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float v = softcap(x[j], p.softcap);
            if ((bits >> j) & 1u) v = penalize(v, p.repetition_penalty);
            pe[j] = expf_glibc_tab((v - vmax) * inv_temp, [&](uint32_t t) { return tab[t]; });
        }
        if (n == 4) {
            *reinterpret_cast<float4*>(pes + i) = make_float4(pe[0], pe[1], pe[2], pe[3]);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                sum += static_cast<double>(pe[j]);
                atomicAdd(&hist_s[fb_bin(pe[j], shift, static_cast<uint32_t>(bins))], 1u);
            }
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (j < n) {
                    pes[i + j] = pe[j];
                    sum += static_cast<double>(pe[j]);
                    atomicAdd(&hist_s[fb_bin(pe[j], shift, static_cast<uint32_t>(bins))], 1u);
                }
            }
        }
    });
    sum = wave::sum_f64(sum);
    if ((tid & 63) == 0) sums[tid >> 6] = sum;
    __syncthreads();
    if (tid == 0) {
        double t = 0.0;
        for (int w = 0; w < kFW; ++w) t += sums[w];
        r.psum[part] = t;
    }
    for (int i = tid; i < bins; i += kFT) {
        const uint32_t c = hist_s[i];
        if (parts == 1) r.bin[i] = c;
        else if (c) atomicAdd(&r.bin[i], c);
    }
}

// Exclusive prefix of one double (count) per thread over the workgroup, and
// the total. The order of the additions is fixed.
__device__ __forceinline__ double fb_scan_f64(double v, double* s, double& total) {
    const int wave = threadIdx.x >> 6;
    const double incl = wave::incl_f64(v);
    if ((threadIdx.x & 63) == 63) s[wave] = incl;
    __syncthreads();
    double before = 0.0;
    total = 0.0;
    for (int w = 0; w < kFW; ++w) {
        if (w == wave) before = total;
        total += s[w];
    }
    __syncthreads();
    return before + (incl - v);
}
__device__ __forceinline__ uint32_t fb_scan_u32(uint32_t v, uint32_t* s, uint32_t& total) {
    const int wave = threadIdx.x >> 6;
    const uint32_t incl = wave::incl_add(v);
    if ((threadIdx.x & 63) == 63) s[wave] = incl;
    __syncthreads();
    uint32_t before = 0;
    total = 0;
    for (int w = 0; w < kFW; ++w) {
        if (w == wave) before = total;
        total += s[w];
    }
    __syncthreads();
    return before + incl - v;
}

// The biased float exponent of x > 0, at least 1 (subnormal floats share the
// first normal binade's ulp); 0 for x <= 0.
__device__ __forceinline__ int fb_expo(double x) {
    if (!(x > 0.0)) return 0;
    return max(static_cast<int>((__builtin_bit_cast(uint64_t, x) >> 52) & 0x7ff) - 1023 + 127, 1);
}
// 1 / ulp of the float binade with biased exponent e.
__device__ __forceinline__ double fb_inv_ulp(int e) { return __builtin_ldexp(1.0, 150 - e); }
// Whether every addend of [lo, hi] adds the same whole number of ulps in the
// binade, none of them a tie.
__device__ __forceinline__ bool fb_alike(float lo, float hi, int e) {
    const double iu = fb_inv_ulp(e);
    const double yl = static_cast<double>(lo) * iu, yh = static_cast<double>(hi) * iu;  // exact
    const double n = __builtin_floor(yh + 0.5);
    return yh < 0x1p24 && yl > n - 0.5 && yh < n + 0.5;
}

// 3. One workgroup per row; thread t holds bins kPer * t .. Latency-bound: five
//    workgroup scans.
template <int kPer>
__global__ __launch_bounds__(kFT) void fb_plan_kernel(DevArgs a, int parts) {
    __shared__ double sd[kFW];
    __shared__ uint32_t su[kFW];
    __shared__ uint32_t smask[kFbMaxBins / 32];
    __shared__ uint32_t s_bad, s_cut, s_stop, s_first, s_last, s_off0, s_off1;
    __shared__ double s_cut_lo, s_cut_hi;
    __shared__ float s_stop_q;
    constexpr int kBins = kPer * kFT;
    const int row = blockIdx.x, tid = threadIdx.x, lane = __lane_id();
    ge_sample_params p;
    if (!fb_serves(a, row, p)) return;
    const int V = a.vocab;
    const FbRow r = fb_row(a, row, kBins);
    uint32_t* meta = fb_meta(a, row);
    uint32_t* pre = a.fo_pre + static_cast<int64_t>(row) * a.fo_items_stride;
    float* aux = a.fo_aux + static_cast<int64_t>(row) * a.fo_items_stride;
    uint64_t* items = a.fo_items + static_cast<int64_t>(row) * a.fo_items_stride;
    const int b0 = tid * kPer;
    uint32_t c[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) c[j] = r.bin[b0 + j];
    float vmax;
    uint32_t shift;
    fb_bin_shape(r, parts, kBins, p, vmax, shift);
    const double S = wave::sum_f64(lane < parts ? r.psum[lane] : 0.0);
    if (tid == 0) {
        s_bad = 0u;
        s_cut = s_stop = s_first = 0xffffffffu;
        s_last = 0u;
        s_cut_lo = s_cut_hi = 0.0;
        s_stop_q = 0.0f;
        s_off0 = s_off1 = 0u;
    }
    for (int i = tid; i < kBins / 32; i += kFT) smask[i] = 0u;
    // The exps of bin b: [lo_bits, hi_bits] (the last bin: from 0).
    auto hi_pe = [&](int j) { return u2f(kOne - (static_cast<uint32_t>(b0 + j) << shift)); };
    auto lo_pe = [&](int j) {
        return b0 + j == kBins - 1 ? 0.0f : u2f(kOne - (static_cast<uint32_t>(b0 + j + 1) << shift) + 1u);
    };
    uint32_t fine = 0, n_t = 0;
    const float tiny = S >= 0.5 && S < 0x1p60 ? __builtin_ldexpf(1.0f, min(sum_exp(S) - 29, 0)) : 1.0f;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        n_t += c[j];
        if (lo_pe(j) < tiny) fine += c[j];
    }
    uint32_t total, n_fine;
    uint32_t before = fb_scan_u32(n_t, su, total);  // elements before this thread's bins
    (void)fb_scan_u32(fine, su, n_fine);
    const float inv_temp = 1.0f / p.temperature;
    const bool fits = inv_temp > 0.0f && inv_temp < __builtin_inff() && vmax > -__builtin_inff() &&
                      vmax < __builtin_inff() && total == static_cast<uint32_t>(V) && den_rounds_alike(S, n_fine, V);
    if (!fits) {  // block-uniform
        if (tid == 0) meta[kMetaStatus] = kStatusToSort;
        return;
    }
    const float inv = static_cast<float>(1.0 / S);
    const float minimum = inv * p.min_p;  // generation.cpp:104, probs[0] = 1 * inv
    const double tp = p.top_p == p.top_p ? static_cast<double>(p.top_p) : 1e30;
    // The min-p cut lies in the first bin with a probability below it.
    {
        uint32_t first = 0xffffffffu;
#pragma unroll
        for (int j = kPer - 1; j >= 0; --j)
            if (c[j] && lo_pe(j) * inv < minimum) first = static_cast<uint32_t>(b0 + j);
        if (first != 0xffffffffu) atomicMin(&s_cut, first);
    }
    // The float sum before each bin: the exact sum first (x0), for the
    // binades, then with every addend rounded as it is there (a0). The bins'
    // own terms are formed again in each sweep, from a copy of inv that the
    // compiler cannot see through: kept, they spill.
    auto mid = [&](int j, float iv) {
        return 0.5 * (static_cast<double>(lo_pe(j) * iv) + static_cast<double>(hi_pe(j) * iv));
    };
    auto rounded = [&](int j, float iv, double acc) {  // bin j's addends in the binade of acc
        const int e = max(fb_expo(acc), 1);
        return c[j] * __builtin_ldexp(__builtin_rint(__builtin_ldexp(mid(j, iv), 150 - e)), e - 150);
    };
    auto opaque = [](float v) {
        asm volatile("" : "+v"(v));
        return v;
    };
    double x0, a0, w0, all;
    {
        double t = 0.0;
        float iv = opaque(inv);
#pragma unroll
        for (int j = 0; j < kPer; ++j) t += c[j] * mid(j, iv);
        x0 = fb_scan_f64(t, sd, all);
        double x = x0;
        t = 0.0;
        iv = opaque(inv);
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const double m = c[j] * mid(j, iv);
            t += rounded(j, iv, x + 0.5 * m);
            x += m;
        }
        a0 = fb_scan_f64(t, sd, all);
    }
    // f(j, inv, the sum before bin j, the sum after it)
    auto sweep = [&](auto&& f) {
        double x = x0, A = a0;
        const float iv = opaque(inv);
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const double m = c[j] * mid(j, iv);
            const double A1 = A + rounded(j, iv, x + 0.5 * m);
            f(j, iv, A, A1);
            x += m;
            A = A1;
        }
    };
    {
        const uint32_t cut = s_cut;  // (written before the scans' barriers)
        sweep([&](int j, float, double A, double A1) {
            const uint32_t b = static_cast<uint32_t>(b0 + j);
            if (b == cut) {
                s_cut_lo = A;
                s_cut_hi = A1;
            }
            if (c[j] && A1 * (1.0 + kFbDrift) >= tp && A * (1.0 + kFbDrift) < tp) atomicMin(&s_stop, b);
        });
        if (cut == 0xffffffffu && tid == 0) s_cut_lo = s_cut_hi = all;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPer; ++j)
        if (static_cast<uint32_t>(b0 + j) == s_stop) s_stop_q = hi_pe(j) * inv;
    __syncthreads();
    const uint32_t cut = s_cut;
    // The mass the draw is taken of: top_p and less than the stopping addend
    // more, or the sum before the cut; at least the first probability.
    const double q_first = static_cast<double>(inv);
    double mass_lo = tp < s_cut_lo ? tp : s_cut_lo;
    const double over = tp + static_cast<double>(s_stop_q);
    double mass_hi = over < s_cut_hi ? over : s_cut_hi;
    if (!(mass_lo > q_first)) {
        mass_lo = q_first;
        mass_hi = max(mass_hi, 2.0 * q_first);
    }
    const double u = static_cast<double>(a.uniforms[row]);
    const double c_lo = u * mass_lo * (1.0 - 2.0 * kFbDrift), c_hi = u * mass_hi * (1.0 + 2.0 * kFbDrift);
    const double c_mid = 0.5 * (c_lo + c_hi);
    // What the walk has taken off before each bin.
    {
        double t = 0.0;
        sweep([&](int j, float iv, double A, double A1) { t += rounded(j, iv, c_mid - 0.5 * (A + A1)); });
        w0 = fb_scan_f64(t, sd, all);
    }
    uint32_t n_items = 0, n_seg = 0;
    uint32_t expand = 0, visit = 0;
    uint32_t tag[kPer];
    uint32_t at = before;
    double W = w0;
    sweep([&](int j, float iv, double A, double A1) {
        const uint32_t b = static_cast<uint32_t>(b0 + j);
        const double W1 = W + rounded(j, iv, c_mid - 0.5 * (A + A1));
        tag[j] = 0u;
        if (c[j] != 0u) {
            const float qh = hi_pe(j) * iv, ql = lo_pe(j) * iv;
            const bool head = at < kFbHead;
            const double a_lo = A * (1.0 - kFbDrift), a_hi = A1 * (1.0 + kFbDrift);
            const bool seen = head || (a_lo < tp && b <= cut);
            bool ex = head || b == cut || a_hi >= tp;
            const int ea = fb_expo(a_lo);
            ex = ex || ea != fb_expo(a_hi) || ea == 0 || !fb_alike(ql, qh, ea);
            tag[j] = static_cast<uint32_t>(ea);
            const double w_hi = c_hi * (1.0 + kFbDrift) - W, w_lo = c_lo - c_hi * kFbDrift - W1;
            if (w_hi > 0.0) {
                const int ew = fb_expo(w_hi);
                if (!(w_lo > 0.0)) {
                    ex = true;
                    if (seen) {  // the walk may stop here
                        atomicMin(&s_first, b);
                        atomicMax(&s_last, b);
                    }
                } else {
                    ex = ex || ew != fb_expo(w_lo) || !fb_alike(ql, qh, ew);
                }
                tag[j] |= static_cast<uint32_t>(ew) << 8;
            }
            if (seen) {
                visit |= 1u << j;
                if (ex) {
                    expand |= 1u << j;
                    n_items += c[j];
                    ++n_seg;
                    if (c[j] > kFbSegMost) s_bad = 1u;
                } else {
                    ++n_items;
                }
            }
        }
        at += c[j];
        W = W1;
    });
    uint32_t G, segs;
    uint32_t off = fb_scan_u32(n_items, su, G);
    uint32_t seg = fb_scan_u32(n_seg, su, segs);
    if (s_bad || static_cast<int64_t>(G) + 1 > fb_half(a) || segs > static_cast<uint32_t>(kFbSegs)) {
        if (tid == 0) meta[kMetaStatus] = kStatusToSort;
        return;
    }
    at = before;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const uint32_t b = static_cast<uint32_t>(b0 + j);
        if ((visit >> j) & 1u) {
            if (b == s_first) s_off0 = off;
            if ((expand >> j) & 1u) {
                r.bin[b] = off;
                r.seg[3 * seg] = off;
                r.seg[3 * seg + 1] = c[j];
                r.seg[3 * seg + 2] = at;
                ++seg;
                off += c[j];
                atomicOr(&smask[b >> 5], 1u << (b & 31u));
            } else {
                items[off] = kFbRegular | tag[j];
                aux[off] = hi_pe(j);
                pre[off] = at;
                ++off;
            }
            if (b == s_last) s_off1 = off;
            if (off == G) pre[G] = at + c[j];
        }
        at += c[j];
    }
    __syncthreads();
    for (int i = tid; i < kBins / 32; i += kFT) r.mask[i] = smask[i];
    if (tid == 0) {
        r.scal[kScShift] = shift;
        r.scal[kScInv] = f2u(inv);
        r.scal[kScDrawBin] = s_first == 0xffffffffu ? 0u : s_first;
        r.scal[kScDrawItem] = s_off0;
        r.scal[kScDrawEnd] = s_first == 0xffffffffu ? 0u : s_off1;
        r.scal[kScSegs] = segs;
        meta[kMetaItems] = G;
        meta[kMetaStatus] = kStatusOk;
    }
}

// 4. The expanded bins' tokens to their items, in no order, and the sum of the
//    probabilities of the bins before the draw's. A streaming read of the
//    exps; about one token in ten is expanded in near-uniform rows.
__global__ __launch_bounds__(kFT) void fb_collect_kernel(DevArgs a) {
    __shared__ uint32_t smask[kFbMaxBins / 32];
    __shared__ double sums[kFW];
    const int row = blockIdx.y, part = blockIdx.x, parts = gridDim.x, tid = threadIdx.x;
    ge_sample_params p;
    if (!fb_serves(a, row, p) || fb_meta(a, row)[kMetaStatus] != kStatusOk) return;
    const int bins = fb_bins(a.vocab);
    const FbRow r = fb_row(a, row, bins);
    for (int i = tid; i < bins / 32; i += kFT) smask[i] = r.mask[i];
    const uint32_t shift = r.scal[kScShift];
    const float inv = u2f(r.scal[kScInv]);
    const uint32_t draw = r.scal[kScDrawBin];
    __syncthreads();
    int lo, hi;
    fb_part(a, part, parts, lo, hi);
    const float* pes = fb_exp_array(a, row);
    uint64_t* items = a.fo_items + static_cast<int64_t>(row) * a.fo_items_stride;
    double sum = 0.0;
    fb_stream<4>(pes, true, lo, hi, tid, [&](int i, float x0, float x1, float x2, float x3, int n) {
        const float x[4] = {x0, x1, x2, x3};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (j < n) {
                const uint32_t b = fb_bin(x[j], shift, static_cast<uint32_t>(bins));
                if (b < draw) sum += static_cast<double>(x[j] * inv);
                if ((smask[b >> 5] >> (b & 31u)) & 1u) {
                    const uint32_t at = atomicAdd(&r.bin[b], 1u);
                    items[at] = (static_cast<uint64_t>(f2u(x[j])) << 32) | (0xffffffffu - static_cast<uint32_t>(i + j));
                }
            }
        }
    });
    sum = wave::sum_f64(sum);
    if ((tid & 63) == 0) sums[tid >> 6] = sum;
    __syncthreads();
    if (tid == 0) {
        double t = 0.0;
        for (int w = 0; w < kFW; ++w) t += sums[w];
        r.pbef[part] = t;
    }
}

// 5. The tokens of each expanded bin by (exp descending, index ascending), with
//    the items' first elements: one wave per bin by counting the larger keys
//    (every lane's up to eight keys against an LDS broadcast), the workgroup
//    by a bitonic sort for the rare larger ones.
constexpr int kOT = 256;
constexpr int kOW = kOT / 64;
__global__ __launch_bounds__(kOT) void fb_order_kernel(DevArgs a) {
    __shared__ uint64_t stage[kFbSegMost];
    static_assert(kOW * kFbWaveSeg <= static_cast<int>(kFbSegMost), "the waves' shares");
    const int row = blockIdx.y, tid = threadIdx.x, lane = __lane_id(), wave = tid >> 6;
    ge_sample_params p;
    if (!fb_serves(a, row, p) || fb_meta(a, row)[kMetaStatus] != kStatusOk) return;
    const FbRow r = fb_row(a, row, fb_bins(a.vocab));
    const int segs = static_cast<int>(r.scal[kScSegs]);
    uint64_t* items = a.fo_items + static_cast<int64_t>(row) * a.fo_items_stride;
    float* aux = a.fo_aux + static_cast<int64_t>(row) * a.fo_items_stride;
    uint32_t* pre = a.fo_pre + static_cast<int64_t>(row) * a.fo_items_stride;
    auto place = [&](uint32_t item, uint32_t elem, uint64_t key) {
        items[item] = key;
        aux[item] = u2f(static_cast<uint32_t>(key >> 32));
        pre[item] = elem;
    };
    uint64_t* mine = stage + wave * kFbWaveSeg;
    bool large = false;
    for (int s = blockIdx.x * kOW + wave; s < segs; s += gridDim.x * kOW) {
        const uint32_t off = r.seg[3 * s], n = r.seg[3 * s + 1], first = r.seg[3 * s + 2];
        if (n <= 64u) {
            const uint64_t key = static_cast<uint32_t>(lane) < n ? items[off + lane] : 0ull;
            uint32_t rank = 0;
            for (uint32_t j = 0; j < n; ++j) rank += wave::readlane64(key, static_cast<int>(j)) > key ? 1u : 0u;
            if (static_cast<uint32_t>(lane) < n) place(off + rank, first + rank, key);
        } else if (n <= static_cast<uint32_t>(kFbWaveSeg)) {
            constexpr int kMy = kFbWaveSeg / 64;
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
                if (static_cast<uint32_t>(v) * 64u + static_cast<uint32_t>(lane) < n) place(off + rank[v], first + rank[v], key[v]);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        } else {
            large = true;
        }
    }
    if (__syncthreads_or(large ? 1 : 0) == 0) return;
    for (int s0 = blockIdx.x * kOW; s0 < segs; s0 += gridDim.x * kOW) {
        for (int s = s0; s < min(s0 + kOW, segs); ++s) {
            const uint32_t off = r.seg[3 * s], n = r.seg[3 * s + 1], first = r.seg[3 * s + 2];
            if (n <= static_cast<uint32_t>(kFbWaveSeg)) continue;  // (block-uniform)
            uint32_t n2 = 1;
            while (n2 < n) n2 <<= 1;
            __syncthreads();
            for (uint32_t i = tid; i < n2; i += kOT) stage[i] = i < n ? items[off + i] : 0ull;
            for (uint32_t size = 2; size <= n2; size <<= 1) {
                for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
                    __syncthreads();
                    for (uint32_t q = tid; q < n2 / 2; q += kOT) {
                        const uint32_t i = 2u * q - (q & (stride - 1u));
                        const uint64_t x = stage[i], y = stage[i + stride];
                        const bool desc = (i & size) == 0u;
                        if (desc ? x < y : x > y) {
                            stage[i] = y;
                            stage[i + stride] = x;
                        }
                    }
                }
            }
            __syncthreads();
            for (uint32_t i = tid; i < n; i += kOT) place(off + i, first + i, stage[i]);
        }
    }
}

// 6. The chains (generation.cpp:103-126) over the items with the whole
//    workgroup, the checks of the plan, and the token. Latency-bound: a pass
//    of block_chain per binade change, most of them 64-item probes at the head.
constexpr int kDrawThreads = 512;
constexpr int kDrawWaves = kDrawThreads / 64;
constexpr int kDrawLog = 96;   // binade changes logged per chain
constexpr int kDrawTies = 4096;  // tokens of one exp (kFbSegMost)

struct DrawShared {
    bchain::Shared<kDrawWaves> bc;
    uint64_t tie[kDrawTies];
    int log_item[kDrawLog];
    uint32_t log_expo[kDrawLog];
    int log_n;
    uint32_t bad;
    double sums[kDrawWaves];
    int32_t token;
};

// Logs the binade that the accumulator is in after each event item.
struct DrawLog {
    DrawShared* sh;
    int n = 0;
    __device__ void operator()(int item, double s) {
        if (threadIdx.x == 0 && n < kDrawLog) {
            sh->log_item[n] = item;
            sh->log_expo[n] = static_cast<uint32_t>(fb_expo(s));
        }
        ++n;
    }
};

__global__ __launch_bounds__(kDrawThreads) void fb_draw_kernel(DevArgs a, int parts) {
    __shared__ DrawShared sh;
    const int row = blockIdx.x, tid = threadIdx.x, lane = __lane_id(), wave = tid >> 6;
    const ge_sample_params pp = a.row_params ? a.row_params[row] : a.params;
    uint32_t k;
    if (!full_order_row(pp, a.vocab, k)) return;
    if (row_done(a, row)) {
        if (tid == 0) skipped_row(a, row);
        return;
    }
    uint32_t* meta = fb_meta(a, row);
    if (meta[kMetaStatus] != kStatusOk) return;  // the sort-based pass serves the row
    const ge_sample_params p = pp;
    const int V = a.vocab;
    const FbRow r = fb_row(a, row, fb_bins(V));
    const int G = static_cast<int>(meta[kMetaItems]);
    const uint64_t* items = a.fo_items + static_cast<int64_t>(row) * a.fo_items_stride;
    const float* aux = a.fo_aux + static_cast<int64_t>(row) * a.fo_items_stride;
    const uint32_t* pre = a.fo_pre + static_cast<int64_t>(row) * a.fo_items_stride;
    const float inv = u2f(r.scal[kScInv]);
    const int draw0 = static_cast<int>(r.scal[kScDrawItem]), draw1 = static_cast<int>(r.scal[kScDrawEnd]);
    if (tid == 0) {
        sh.bad = 0u;
        sh.token = -1;
    }
    const float q0 = aux[0] * inv;
    const float minimum = q0 * p.min_p;
    const uint32_t end = pre[G];
    // generation.cpp:106-108: the first element e >= 1 with p_e < minimum.
    uint32_t keff = static_cast<uint32_t>(V);
    if (q0 < minimum) {
        keff = 1u;
    } else if (minimum > 0.0f && G > 1) {
        const uint32_t pq = wave_partition_point(1u, static_cast<uint32_t>(G), [&](uint32_t i) { return !(aux[i] * inv < minimum); });
        if (pq < static_cast<uint32_t>(G)) keff = pre[pq];
    }
    __syncthreads();
    // Whether every item before `last` that stands for a bin was passed in the
    // binade the plan took it in (tag bits 0-7 for the cumulative, 8-15 for the
    // walk), and no event fell on one.
    auto check = [&](int n_log, int last, uint32_t first_expo, int shift) {
        __syncthreads();  // the log is written
        if (n_log > kDrawLog && tid == 0) sh.bad = 1u;
        const int n = min(n_log, kDrawLog);
        for (int i = tid; i < last; i += kDrawThreads) {
            const uint64_t it = items[i];
            if (!(it & kFbRegular)) continue;
            uint32_t e = first_expo;
            bool hit = false;
            for (int l = 0; l < n; ++l) {
                const int li = sh.log_item[l];
                if (li < i) e = sh.log_expo[l];
                hit = hit || li == i;
            }
            if (hit || ((static_cast<uint32_t>(it) >> shift) & 0xffu) != e) sh.bad = 1u;
        }
        __syncthreads();
    };
    auto expanded = [&](int i) { return i >= 0 && i < G && !(items[i] & kFbRegular); };
    uint32_t pos = 0;
    int item = 0;
    bool ok = true, near = false;
    {
        double s = static_cast<double>(q0);
        ChainPos cp{0, 1};
        uint32_t keep = keff;
        if (keff > 1u) {
            const uint32_t L = min(keff, end);
            DrawLog log{&sh};
            const bool hit = L > 1u && bchain::block_chain<bchain::F32Acc, false, kDrawThreads>(
                                           pre, aux, inv, G, cp, L, s, static_cast<double>(p.top_p), sh.bc, log);
            if (hit) keep = cp.elem + 1u;
            else if (L < keff) ok = false;  // the plan's items end before the cut
            check(log.n, min(cp.item + 1, G), static_cast<uint32_t>(fb_expo(static_cast<double>(q0))), 0);
        }
        const float mass = static_cast<float>(s);
        const float u = a.uniforms[row];
        const float choice = u * (mass - 0.0f) + 0.0f;  // random.h:1864-1871
        if (ok && choice > 0.0f && choice < __builtin_inff()) {
            ChainPos w{0, 0};
            double c = static_cast<double>(choice);
            DrawLog log{&sh};
            const bool stop = bchain::block_chain<bchain::F32Acc, true, kDrawThreads>(pre, aux, inv, G, w, min(keep, end), c,
                                                                                     0.0, sh.bc, log);
            pos = stop ? w.elem : keep - 1u;
            item = w.item;
            check(log.n, min(item + 1, G), static_cast<uint32_t>(fb_expo(static_cast<double>(choice))), 8);
        } else if (!(choice <= 0.0f)) {
            ok = false;
        }
        ok = ok && expanded(item) && sh.bad == 0u;
        if (ok) {
            // Near-boundary flag: double sums of the probabilities before and
            // through the chosen position; the sum before the draw's bins is
            // fb_collect's, the rest its single tokens.
            double before = 0.0;
            bool nb = false, na = false;
            const double ch = static_cast<double>(choice);
            bool sure = true;
            if (pos > 0u) {
                if (item < draw0 || item >= draw1) {
                    sure = false;
                } else {
                    double t = 0.0;
                    for (int i = draw0 + tid; i < item; i += kDrawThreads) t += static_cast<double>(aux[i] * inv);
                    t = wave::sum_f64(t);
                    if (lane == 0) sh.sums[wave] = t;
                    __syncthreads();
                    before = wave::sum_f64(lane < parts ? r.pbef[lane] : 0.0);
                    for (int v = 0; v < kDrawWaves; ++v) before += sh.sums[v];
                    sure = near_decided(ch, before, near_sum_error(pos), nb);
                }
            }
            sure = sure && near_decided(ch, before + static_cast<double>(aux[item] * inv), near_sum_error(pos), na);
            near = (pos > 0u && nb) || (pos + 1u < keep && na);
            ok = sure;
        }
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
    if (n_tie == 1) {
        if (tid == 0) sh.token = static_cast<int32_t>(composite_index(items[item]));
    } else {  // (at most kFbSegMost: one exp lies in one bin)
        for (int i = tid; i < n_tie; i += kDrawThreads) {
            const uint32_t idx = composite_index(items[is + i]);
            float v = softcap(rowp[idx], p.softcap);
            if (pen && ((bitmap[idx >> 5] >> (idx & 31u)) & 1u)) v = penalize(v, p.repetition_penalty);
            sh.tie[i] = composite(order_key(v), idx);
        }
        __syncthreads();
        const uint32_t want = static_cast<uint32_t>(item - is);
        for (int i = tid; i < n_tie; i += kDrawThreads) {
            const uint64_t x = sh.tie[i];
            uint32_t rank = 0;
            for (int j = 0; j < n_tie; ++j) rank += sh.tie[j] > x ? 1u : 0u;
            if (rank == want) sh.token = static_cast<int32_t>(composite_index(x));
        }
    }
    __syncthreads();
    // The bitmap is all zero again after every call (cleared from the history
    // before the token is appended: a full ring's history is the ring).
    if (pen) {
        for (int i = tid; i < H; i += kDrawThreads) {
            const int32_t id = hist[i];
            if (id >= 0 && id < V) bitmap[id >> 5] = 0u;
        }
        __syncthreads();
    }
    if (tid == 0) emit_row(a, row, sh.token, aux[item] * inv, near ? GE_FLAG_NEAR_BOUNDARY : 0);
}

}  // namespace

hipError_t launch_binned(const DevArgs& a, hipStream_t stream) {
    // Parts per row: about two workgroups per CU in all, at most one per step.
    const int steps = (a.vocab + kFStep - 1) / kFStep;
    const int parts = std::max(1, std::min({steps, kFbParts, (512 + a.rows - 1) / a.rows}));
    const dim3 grid(static_cast<unsigned>(parts), static_cast<unsigned>(a.rows));
    const int bins = fb_bins(a.vocab);
    hipLaunchKernelGGL(fb_range_kernel, grid, dim3(kFT), 0, stream, a);
    hipLaunchKernelGGL(fb_exps_kernel, grid, dim3(kFT), 0, stream, a);
    const dim3 rows(static_cast<unsigned>(a.rows));
    switch (bins / kFT) {
        case 2: hipLaunchKernelGGL(fb_plan_kernel<2>, rows, dim3(kFT), 0, stream, a, parts); break;
        case 4: hipLaunchKernelGGL(fb_plan_kernel<4>, rows, dim3(kFT), 0, stream, a, parts); break;
        case 8: hipLaunchKernelGGL(fb_plan_kernel<8>, rows, dim3(kFT), 0, stream, a, parts); break;
        default: hipLaunchKernelGGL(fb_plan_kernel<16>, rows, dim3(kFT), 0, stream, a, parts); break;
    }
    hipLaunchKernelGGL(fb_collect_kernel, grid, dim3(kFT), 0, stream, a);
    const unsigned ob = static_cast<unsigned>(std::max(4, std::min(128, 2048 / a.rows)));
    hipLaunchKernelGGL(fb_order_kernel, dim3(ob, static_cast<unsigned>(a.rows)), dim3(kOT), 0, stream, a);
    hipLaunchKernelGGL(fb_draw_kernel, rows, dim3(kDrawThreads), 0, stream, a, parts);
    return hipGetLastError();
}

}  // namespace ge
