// log2_math.hpp -- FP32 log2 through FP64, rounded once: the to_decibels kernel and the FP32 fused
// launch share it, so both give the same bits.
#pragma once

#include <hip/hip_runtime.h>

namespace rppa {

// log2(x) for x > 0 (subnormal and infinite x included).  With x = f 2^e, f in [sqrt(1/2), sqrt(2)), and
// s = (f - 1) / (f + 1): log2 f = 2 / ln 2 (s + s^3 / 3 + ... + s^19 / 19), |s| <= 0.1716, so the terms
// left out are below 2^-54 of the result, and the FP64 sum is within 2^-50 of it: the rounding to FP32
// differs from the correctly rounded value only within 2^-26 ulp of a tie.  About 25 FP64 operations
// against some 90 of the library's log2 (which serves every double).
__device__ __forceinline__ float log2_rn(float x)
{
    const double d = static_cast<double>(x);
    double f = __builtin_amdgcn_frexp_mant(d);      // [0.5, 1)
    int e = __builtin_amdgcn_frexp_exp(d);
    const bool low = f < 0.70710678118654752;
    f = low ? f + f : f;
    e = low ? e - 1 : e;
    const double n = f - 1.0, m = f + 1.0;          // exact: f has 24 bits
    double r = __builtin_amdgcn_rcp(m);             // two Newton steps from the 2^-14 or better estimate
    r = fma(fma(-m, r, 1.0), r, r);
    r = fma(fma(-m, r, 1.0), r, r);
    double s = n * r;
    s = fma(fma(-m, s, n), r, s);
    const double z = s * s;
    double p = 0.15186263588304877;
    p = fma(p, z, 0.16972882833987804);
    p = fma(p, z, 0.19235933878519512);
    p = fma(p, z, 0.22195308321368667);
    p = fma(p, z, 0.26230818925253879);
    p = fma(p, z, 0.3205988979753252);
    p = fma(p, z, 0.41219858311113239);
    p = fma(p, z, 0.57707801635558531);
    p = fma(p, z, 0.96179669392597555);
    p = fma(p, z, 2.8853900817779268);
    const double v = fma(p, s, static_cast<double>(e));
    return x < __builtin_inff() ? static_cast<float>(v) : x;
}

}  // namespace rppa
