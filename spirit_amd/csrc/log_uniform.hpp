// The logarithm of a uniform random number.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

namespace spirit_hip
{

// log u of a uniform u in (0, 1], u a multiple of 2^-53: no infinities, denormals or negative
// arguments to sort out.  With u = m 2^k, m in [sqrt(1/2), sqrt(2)), f = m - 1 and s = f / (2 + f),
// log m = 2 artanh s = f - s (f - 2 (s^2/3 + s^4/5 + ...)); s^2 <= 0.0295, the first omitted term,
// 2 s s^20 / 21, is below 2.8e-17 of f.  s itself counts only by a sixth of f, so a reciprocal with two
// Newton steps is enough for it: rcp( d ) is 1 / d to 2^-23.  At most 1.1 units in the last place off.
template<typename RCP>
__device__ __forceinline__ double log_uniform( double u, RCP rcp )
{
    int k;
    double m       = frexp( u, &k );
    const bool low = m < 0.70710678118654752;
    m              = low ? m + m : m;
    k              = low ? k - 1 : k;
    const double f = m - 1.0, d = 2.0 + f;
    double r       = rcp( d );
    r              = fma( fma( -d, r, 1.0 ), r, r );
    r              = fma( fma( -d, r, 1.0 ), r, r );
    const double s = f * r, z = s * s;
    double p       = 1.0 / 19.0;
    p              = fma( p, z, 1.0 / 17.0 );
    p              = fma( p, z, 1.0 / 15.0 );
    p              = fma( p, z, 1.0 / 13.0 );
    p              = fma( p, z, 1.0 / 11.0 );
    p              = fma( p, z, 1.0 / 9.0 );
    p              = fma( p, z, 1.0 / 7.0 );
    p              = fma( p, z, 1.0 / 5.0 );
    p              = fma( p, z, 1.0 / 3.0 );
    // ln 2 as its nearest double and the rest; t holds k ln 2 + f, w what its roundings left
    const double kd = (double)k;
    const double t  = fma( kd, 0.69314718055994531, f );
    const double w  = fma( kd, 0.69314718055994531, f - t );
    return t + ( w - fma( s, f - 2.0 * ( p * z ), -kd * 2.3190468138462996e-17 ) );
}

} // namespace spirit_hip
