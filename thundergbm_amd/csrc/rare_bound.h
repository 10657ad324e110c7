// What the filter of the rare features knows of a row (sparse_kernels.hip, k_sparse_rare_filter), and the range that the
// sums of a candidate lie in by it. Plain arithmetic, for the device and for a test on the host.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>

#include "common.h"

namespace tgbm {
namespace {

// row word: node of the level (11 bits, all ones: the row has come to rest above), sign of g, |g| (10 bits, rounded up), h
// (10 bits, rounded down), both in kRareSteps steps of the tree's largest
constexpr unsigned kRareNodeMask = 0x7ffu;
constexpr float kRareSteps = 1022.f;
// g, h: the integers that the sums are made of; gq_max, hq_max: the tree's largest
__host__ __device__ inline unsigned rare_word(unsigned node, float g, float h, float gq_max, float hq_max) {
    const float a = fabsf(g);
    const unsigned ug = a > 0.f ? (unsigned)ceilf(a * (kRareSteps / gq_max)) : 0u, cg = ug < 1023u ? ug : 1023u;
    const unsigned uh = h > 0.f ? (unsigned)(h * (kRareSteps / hq_max)) : 0u, ch = uh < 1023u ? uh : 1023u;
    return node | (g < 0.f ? 1u << 11 : 0u) | cg << 12 | ch << 22;
}

struct RareCell {
    unsigned long long g;  // sums of the positive g (22 bits) and of the negative g (22), values (13)
    unsigned h;            // sum of h
    __host__ __device__ int plus() const { return (int)((unsigned)g & 0x3fffffu); }
    __host__ __device__ int minus() const { return (int)((unsigned)(g >> 22) & 0x3fffffu); }
    __host__ __device__ int values() const { return (int)(g >> 44); }
};
__host__ __device__ inline RareCell operator+(RareCell a, RareCell b) { return {a.g + b.g, a.h + b.h}; }
__host__ __device__ inline RareCell operator-(RareCell a, RareCell b) { return {a.g - b.g, a.h - b.h}; }
__host__ __device__ inline unsigned long long rare_addend(unsigned word) {
    const unsigned long long g = (word >> 12) & 0x3ffu;
    return 1ull << 44 | ((word >> 11 & 1u) ? g << 22 : g);
}

struct RareBound {
    float g, h, mcw, lambda;  // one step of g and of h
};
struct RareRange {
    float g_min, g_max, h_min, h_max;
};

// Sums of all of `whole` and some of the values of `part`. A code is off by less than a step and, as a rounded float, by
// 2^-22 of itself: the steps (and 2^-22 of terms that cancel) are in the slack of a value of `whole`, what is relative to
// a sum moves its end outwards, away from the other one - whichever sign the end has.
__host__ __device__ inline RareRange rare_range(RareCell whole, RareCell part, RareBound u) {
    constexpr float wide = 0x1p-12f;
    const float base = (float)(whole.plus() - whole.minus()), slack = 1.01f * (float)whole.values();
    const float hi = (base + slack + (float)part.plus()) * u.g, lo = (base - slack - (float)part.minus()) * u.g;
    RareRange r;
    r.g_max = hi + fabsf(hi) * wide;
    r.g_min = lo - fabsf(lo) * wide;
    r.h_min = (float)whole.h * u.h * (1.f - wide);
    r.h_max = (float)((int)(whole.h + part.h) + whole.values() + part.values()) * u.h * (1.f + wide);
    return r;
}

}  // namespace
}  // namespace tgbm
