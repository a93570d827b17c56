// FP64 complex arithmetic and the small power-of-two DFTs of the transforms.
#pragma once

#include "device_types.hpp"

namespace spirit_hip
{

__device__ __forceinline__ double2 cmul( double2 a, double2 b )
{
    return make_double2( a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x );
}
__device__ __forceinline__ double2 cadd( double2 a, double2 b )
{
    return make_double2( a.x + b.x, a.y + b.y );
}
__device__ __forceinline__ double2 csub( double2 a, double2 b )
{
    return make_double2( a.x - b.x, a.y - b.y );
}
__device__ __forceinline__ double2 cconj( double2 a )
{
    return make_double2( a.x, -a.y );
}
// multiply by -i (forward) or +i (inverse)
template<bool INV>
__device__ __forceinline__ double2 mul_mi( double2 a )
{
    return INV ? make_double2( -a.y, a.x ) : make_double2( a.y, -a.x );
}

// unnormalised DFT of R = 2, 4 or 8 values in registers
template<int R, bool INV>
__device__ __forceinline__ void dft_small( double2 * v )
{
    static_assert( R == 2 || R == 4 || R == 8, "" );
    if constexpr( R == 2 )
    {
        double2 a = v[0], b = v[1];
        v[0]      = cadd( a, b );
        v[1]      = csub( a, b );
    }
    else if constexpr( R == 4 )
    {
        double2 a0 = cadd( v[0], v[2] ), a1 = csub( v[0], v[2] );
        double2 b0 = cadd( v[1], v[3] ), b1 = mul_mi<INV>( csub( v[1], v[3] ) );
        v[0]       = cadd( a0, b0 );
        v[2]       = csub( a0, b0 );
        v[1]       = cadd( a1, b1 );
        v[3]       = csub( a1, b1 );
    }
    else if constexpr( R == 8 )
    {
        // DIT: even/odd radix-4 halves, then the w8^k combination.
        double2 e[4] = { v[0], v[2], v[4], v[6] };
        double2 o[4] = { v[1], v[3], v[5], v[7] };
        dft_small<4, INV>( e );
        dft_small<4, INV>( o );
        const double h = 0.70710678118654752440084436210484903928483593768847;
        // w8^1 = (1 -+ i)/sqrt2, w8^2 = -+i, w8^3 = (-1 -+ i)/sqrt2
        double2 t1 = INV ? make_double2( h * ( o[1].x - o[1].y ), h * ( o[1].x + o[1].y ) )
                         : make_double2( h * ( o[1].x + o[1].y ), h * ( o[1].y - o[1].x ) );
        double2 t2 = mul_mi<INV>( o[2] );
        double2 t3 = INV ? make_double2( -h * ( o[3].x + o[3].y ), h * ( o[3].x - o[3].y ) )
                         : make_double2( h * ( o[3].y - o[3].x ), -h * ( o[3].x + o[3].y ) );
        v[0] = cadd( e[0], o[0] );
        v[4] = csub( e[0], o[0] );
        v[1] = cadd( e[1], t1 );
        v[5] = csub( e[1], t1 );
        v[2] = cadd( e[2], t2 );
        v[6] = csub( e[2], t2 );
        v[3] = cadd( e[3], t3 );
        v[7] = csub( e[3], t3 );
    }
}

} // namespace spirit_hip
