// Small device helpers shared by the kernel sources (wave64 indexing, 64-bit shuffles, the reference's gain
// formula and left/right rule). Everything here is inlined into its callers.
#pragma once
#include <hip/hip_runtime.h>

#include "device_api.h"

namespace tgbm {
namespace {

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }
__device__ __forceinline__ int wave_id() { return threadIdx.x >> 6; }
__device__ __forceinline__ int lanes_below(unsigned long long mask) {
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0));
}


// Round-to-nearest-even of a float (|x| < 2^51) as a 64-bit integer: the integer sits in the low mantissa bits of
// x + 1.5 * 2^52 (bit pattern 0x4338000000000000, whose low word is zero: only the high word is corrected).
__device__ __forceinline__ long long round_to_ll(float x) {
    const long long b = __double_as_longlong((double)x + 6755399441055744.0);
    const unsigned hi = (unsigned)((unsigned long long)b >> 32) - 0x43380000u;
    return (long long)(((unsigned long long)hi << 32) | (unsigned)b);
}

__device__ __forceinline__ bool node_splits(const TreeNode &nd) {
    return nd.is_valid && !nd.is_leaf && nd.split_feature_id >= 0;
}


// Scans and reductions over a wavefront move values between lanes with DPP, a modifier of vector instructions: a few cycles
// a step, where __shfl goes through the LDS crossbar and the wavefront waits about 0.1 us for each. What they are used for
// are chains that a whole launch waits for: the split search of a pack took 3.2 us with twelve rounds of dependent shuffles in
// it, 2.05 without (500 k x 28, inside a launch of 7.7 and 6.7 us), planning a histogram item 1.6 and 1.1. Every lane of the
// wavefront has to be active.
// Lanes without a source lane, and those outside ROWS (one bit per 16 lanes), get `old`.
constexpr int kDppRowShr = 0x110;    // + n: from the lane n below, within 16 lanes
constexpr int kDppWaveShr1 = 0x138;  // from the lane below
constexpr int kDppBcast15 = 0x142;   // lane 15 of every 16 to the next 16 lanes
constexpr int kDppBcast31 = 0x143;   // lane 31 to lanes 32 .. 63
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ int dpp_i(int old, int v) {
    return __builtin_amdgcn_update_dpp(old, v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ long long dpp_ll(long long v) {  // (0 where there is no source)
    const int lo = dpp_i<CTRL, ROWS>(0, (int)(unsigned)(unsigned long long)v);
    const int hi = dpp_i<CTRL, ROWS>(0, (int)((unsigned long long)v >> 32));
    return (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}
// step.template at<CTRL, ROWS>() for the six steps of an inclusive scan: lane i then holds what lanes 0 .. i held
template <typename Step>
__device__ __forceinline__ void wave_scan_steps(Step &step) {
    step.template at<kDppRowShr + 1, 0xf>();
    step.template at<kDppRowShr + 2, 0xf>();
    step.template at<kDppRowShr + 4, 0xf>();
    step.template at<kDppRowShr + 8, 0xf>();
    step.template at<kDppBcast15, 0xa>();
    step.template at<kDppBcast31, 0xc>();
}

__device__ __forceinline__ long long shfl_up_ll(long long v, int d) {
    int lo = __shfl_up((int)(unsigned)(unsigned long long)v, d);
    int hi = __shfl_up((int)((unsigned long long)v >> 32), d);
    return (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

__device__ __forceinline__ int read_lane(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }  // (uniform lane)
__device__ __forceinline__ float read_lane(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ long long read_lane_ll(long long v, int lane) {
    const unsigned lo = (unsigned)read_lane((int)(unsigned)(unsigned long long)v, lane);
    const unsigned hi = (unsigned)read_lane((int)((unsigned long long)v >> 32), lane);
    return (long long)(((unsigned long long)hi << 32) | lo);
}

// Inclusive sums of two 64-bit integers over a wavefront: four additions a step, the lane move part of them. The compiler does not
// look for hazards inside: a carry may be read one wait state after the vector instruction that writes it, a register through
// DPP two after it was written (between the steps there are more, before the first one there is an s_nop), a lane one after.
__device__ __forceinline__ void wave_scan_pair(long long &a, long long &b) {
    unsigned al = (unsigned)(unsigned long long)a, ah = (unsigned)((unsigned long long)a >> 32);
    unsigned bl = (unsigned)(unsigned long long)b, bh = (unsigned)((unsigned long long)b >> 32);
#define TGBM_SCAN_STEP(MOVE)                           \
    "v_add_co_u32_dpp %0, vcc, %0, %0 " MOVE "\n"      \
    "s_nop 0\n"                                        \
    "v_addc_co_u32_dpp %1, vcc, %1, %1, vcc " MOVE "\n" \
    "v_add_co_u32_dpp %2, vcc, %2, %2 " MOVE "\n"      \
    "s_nop 0\n"                                        \
    "v_addc_co_u32_dpp %3, vcc, %3, %3, vcc " MOVE "\n"
    asm("s_nop 1\n"
        TGBM_SCAN_STEP("row_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:0")
        TGBM_SCAN_STEP("row_shr:2 row_mask:0xf bank_mask:0xf bound_ctrl:0")
        TGBM_SCAN_STEP("row_shr:4 row_mask:0xf bank_mask:0xf bound_ctrl:0")
        TGBM_SCAN_STEP("row_shr:8 row_mask:0xf bank_mask:0xf bound_ctrl:0")
        TGBM_SCAN_STEP("row_bcast:15 row_mask:0xa bank_mask:0xf")
        TGBM_SCAN_STEP("row_bcast:31 row_mask:0xc bank_mask:0xf")
        "s_nop 0\n"
        : "+v"(al), "+v"(ah), "+v"(bl), "+v"(bh) : : "vcc");
#undef TGBM_SCAN_STEP
    a = (long long)((unsigned long long)ah << 32 | al);
    b = (long long)((unsigned long long)bh << 32 | bl);
}

struct WaveSumI {
    int v;
    template <int CTRL, int ROWS>
    __device__ __forceinline__ void at() { v += dpp_i<CTRL, ROWS>(0, v); }
};
struct WaveSumLL {
    long long v;
    template <int CTRL, int ROWS>
    __device__ __forceinline__ void at() { v += dpp_ll<CTRL, ROWS>(v); }
};
struct WaveMaxF {
    float v;
    template <int CTRL, int ROWS>
    __device__ __forceinline__ void at() {
        const int i = __float_as_int(v);
        v = fmaxf(v, __int_as_float(dpp_i<CTRL, ROWS>(i, i)));
    }
};
struct WaveMinI {
    int v;
    template <int CTRL, int ROWS>
    __device__ __forceinline__ void at() { v = min(v, dpp_i<CTRL, ROWS>(v, v)); }
};
__device__ __forceinline__ int wave_scan_i(int v) {  // inclusive
    WaveSumI s{v};
    wave_scan_steps(s);
    return s.v;
}
__device__ __forceinline__ long long wave_scan_ll(long long v) {  // inclusive
    WaveSumLL s{v};
    wave_scan_steps(s);
    return s.v;
}
// (the same in every lane, as scalars)
__device__ __forceinline__ int wave_sum_i(int v) { return read_lane(wave_scan_i(v), 63); }
__device__ __forceinline__ long long wave_sum_ll(long long v) { return read_lane_ll(wave_scan_ll(v), 63); }
__device__ __forceinline__ float wave_max_f(float v) {
    WaveMaxF s{v};
    wave_scan_steps(s);
    return read_lane(s.v, 63);
}
__device__ __forceinline__ int wave_min_i(int v) {
    WaveMinI s{v};
    wave_scan_steps(s);
    return read_lane(s.v, 63);
}
// The lane with the largest v, among equal ones the first with the smallest index; the same in every lane. v is no NaN.
__device__ __forceinline__ int wave_best(float v, int idx, float *win, int *win_idx) {
    *win = wave_max_f(v);
    const bool top = v == *win;
    *win_idx = wave_min_i(top ? idx : 0x7fffffff);
    return __ffsll((long long)__ballot(top && idx == *win_idx)) - 1;
}


// A row's gradient pair from the word (word_from_row).
__device__ __forceinline__ GHPair pair_from_word(int objective, unsigned w) {
    GHPair o;
    if (objective == OBJ_SQUARE) {
        o.g = __uint_as_float(w);
        o.h = 1.f;
    } else {
        const float s = __uint_as_float(w & 0x7fffffffu);
        const float yi = (w >> 31) ? 1.f : 0.f;
        o.g = s - yi;
        o.h = fmaxf(s * (1.f - s), 1e-16f);
    }
    return o;
}


// Left/right decision of the sparse layout: binary search of the row's bin ids for the one inside
// the split feature's bin range (absent = missing), hist_tree_builder_single.cu:941-1011.
// Does the row go right at a split of the feature whose global bins are [cb, ce)? Binary search of the
// row's ascending bin ids for one inside the feature's range; none = missing -> default direction.
__device__ __forceinline__ bool csr_goes_right(const CsrBins &bins, int row, int cb, int ce, int sbid, bool dr) {
    int lo = bins.row_ptr[row], hi = bins.row_ptr[row + 1];
    int found = -1;
    while (lo < hi) {
        int mid = lo + (hi - lo) / 2;
        int b = bins.bin[mid];
        if (b >= cb && b < ce) {
            found = b;
            break;
        }
        if (b < cb)
            lo = mid + 1;
        else
            hi = mid;
    }
    return found < 0 ? dr : (found >= sbid);
}


// Power of two by which the dense work items of a node that add at most `rows` rows between two drains coarsen one
// of the tree's scales: the smallest s >= 0 with rows * (qmax / 2^s + 0.5) < 2^bits (qmax: the most one row adds at the tree's
// scale, bits: magnitude bits of the packed field).
__device__ __forceinline__ int item_shift(float qmax, int rows, int bits) {
    const double lim = ldexp(1.0, bits) / (double)rows * (1.0 - 1e-6) - 0.5;
    const double q = (double)qmax;
    if (!(q >= lim)) return 0;
    return ilogb(q / lim) + 1;  // 2^s > q / lim
}

// ------------------------------------------------------------------------ split finding
// (float)((double)v * inv), inv a power of two: the integer's halves are scaled exactly and added with one rounding.
__device__ __forceinline__ float scaled_float(long long v, double inv) {
    const double hi = (double)(int)(v >> 32), lo = (double)(unsigned)(unsigned long long)v;
    return (float)__fma_rn(hi, inv * 4294967296.0, lo * inv);
}

// split_gain without a branch; fterm: (f.g * f.g) / (f.h + lambda)
__device__ __forceinline__ float split_gain_select(GHPair f, float fterm, GHPair l, float mcw, float lambda) {
#pragma clang fp contract(off)
    const GHPair r{f.g - l.g, f.h - l.h};
    const float gain = (l.g * l.g) / (l.h + lambda) + (r.g * r.g) / (r.h + lambda) - fterm;
    return fmaxf(0.f, ((l.h >= mcw) & (r.h >= mcw)) ? gain : 0.f);
}
__device__ __forceinline__ float split_gain(GHPair f, GHPair l, float mcw, float lambda) {
#pragma clang fp contract(off)
    GHPair r{f.g - l.g, f.h - l.h};
    float gain = 0.f;
    if (l.h >= mcw && r.h >= mcw)
        gain = (l.g * l.g) / (l.h + lambda) + (r.g * r.g) / (r.h + lambda) - (f.g * f.g) / (f.h + lambda);
    return fmaxf(0.f, gain);
}



}  // namespace
}  // namespace tgbm
