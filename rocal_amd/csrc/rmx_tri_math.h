// Coordinate and coefficient law of the triangular (antialiased) resize, shared by its kernels. Every function is the
// fp32 arithmetic of the reference's device kernel, operation for operation (rocal_hip_kernels.cpp:487-589).
#pragma once
#include "rmx_device.h"

namespace rmx {

struct TriAxis {
    float ratio, radius, fscale, offset;
    int ksize;
};

RMX_DEV TriAxis tri_axis(float ratio, float fscale) {
    TriAxis t;
    t.ratio = ratio;
    t.radius = ratio > 1.0f ? ratio : 1.0f;
    t.fscale = fscale;
    t.offset = (ratio - 1) * 0.5f - t.radius;
    t.ksize = (int)ceilf(t.radius * 2);
    return t;
}

RMX_DEV void tri_loc(const TriAxis &t, int d, float lo, int &loc, float &w0) {
    float raw = (float)d * t.ratio;
    raw = raw + t.offset;
    raw = raw + lo;
    loc = (int)ceilf(raw);
    w0 = (float)loc - raw;
}

RMX_DEV float tri_coeff(float w0, float radius, int k, float fscale) {
    float c = 1 - fabsf((w0 - radius + (float)k) * fscale);
    return __builtin_fmaxf(c, 0.0f);  // (c < 0 ? 0 : c, for a c that is a number: ratios are finite)
}

// 1 / b correctly rounded, for the products of coefficient sums (b far from the ends of the exponent range): the hardware's
// reciprocal and one correction by its remainder (Markstein, IBM J. Res. Dev. 34, 1990), three instructions where the division is ten.
// An estimate within an ulp is corrected for every significand but that of all ones, where the power of two next to 1 / b would stay as it
// is: that the hardware does not answer with it is its own doing. tests/test_gpu_reciprocals.py runs through every significand at
// every exponent from -40 to 40.
RMX_DEV float recip(float b) {
    const float y = __builtin_amdgcn_rcpf(b);
    return __builtin_fmaf(__builtin_fmaf(-b, y, 1.0f), y, y);
}

}  // namespace rmx
