// Mixed-radix Stockham FFT over a tile of lines for any length with prime factors up to 13
// (FP64 complex), for gfx950.
//
// A tile holds nl lines of n points, line index fastest: point p of line l lives in LDS at
// [p * lsr + l], so neighbouring lanes work on neighbouring lines of the same point and both the
// LDS accesses and the global accesses of column passes are contiguous whatever the radix is.
// m threads share a line (thread t: line t mod nl, butterflies t / nl, t / nl + m, ...), so a
// thread's line, and with it its addresses, is the same in every stage.
// The first stage takes its inputs from a load functor (global memory) and the last one hands its
// outputs to a store functor, so a transform of S stages crosses LDS S - 1 times.  Stages are
// radix 2 to 10, and 11 to 13 where the length has a factor 11 or 13 (MixPlan; chosen for few
// stages first): each butterfly sits in one thread's
// registers, and the radix of a stage is a uniform branch.  Stages between the first and the last
// run in place: every thread reads all its butterflies' inputs before a barrier and writes the
// outputs after it.
//
// Stage twiddles w_n^(r jm n/(Ns R)) come from a table in stage order, [r - 1][jm], which the
// block copies to LDS behind its tile (or reads where it is): the lanes that share jm read one address.
#pragma once

#include "fft_small.hpp"

namespace spirit_hip
{

// floor(x / d) for 0 <= x < 2^14 and the reciprocal of d < 2^13 in f: (x + 1/2) / d is at least
// 1/(2 d) from a whole number, more than the three roundings of its value (below 2^14 / d) move it
__device__ __forceinline__ int mix_div( int x, const MixDiv & f )
{
    return (int)( ( (float)x + 0.5f ) * f.inv );
}

// odd primes: X[k] = v0 + sum_r cos(2 pi k r / R) (v[r] + v[R-r]) -+ i sum_r sin(2 pi k r / R) (v[r] - v[R-r])
template<int R>
struct OddRoots;
template<>
struct OddRoots<3>
{
    static constexpr double c[1] = { -0.5 };
    static constexpr double s[1] = { 0.86602540378443864676 };
};
template<>
struct OddRoots<5>
{
    static constexpr double c[2] = { 0.30901699437494742410, -0.80901699437494742410 };
    static constexpr double s[2] = { 0.95105651629515357212, 0.58778525229247312917 };
};
template<>
struct OddRoots<7>
{
    static constexpr double c[3] = { 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624 };
    static constexpr double s[3] = { 0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048 };
};
template<>
struct OddRoots<11>
{
    static constexpr double c[5] = { 0.84125353283118116886, 0.41541501300188642553, -0.14231483827328514044,
                                     -0.65486073394528506406, -0.95949297361449738989 };
    static constexpr double s[5] = { 0.54064081745559758211, 0.90963199535451837141, 0.98982144188093273238,
                                     0.75574957435425828377, 0.28173255684142969771 };
};
template<>
struct OddRoots<13>
{
    static constexpr double c[6] = { 0.88545602565320989590, 0.56806474673115580251, 0.12053668025532305335,
                                     -0.35460488704253562597, -0.74851074817110109863, -0.97094181742605202716 };
    static constexpr double s[6] = { 0.46472317204376854566, 0.82298386589365639458, 0.99270887409805399280,
                                     0.93501624268541482344, 0.66312265824079520238, 0.23931566428755776715 };
};

template<int R, bool INV>
__device__ __forceinline__ void dft_odd( double2 * v )
{
    constexpr int H = ( R - 1 ) / 2;
    double2 a[H], b[H]; // sums and differences of the pairs r, R - r
#pragma unroll
    for( int r = 1; r <= H; ++r )
    {
        a[r - 1] = cadd( v[r], v[R - r] );
        b[r - 1] = csub( v[r], v[R - r] );
    }
    const double2 v0 = v[0];
    double2 t        = v0;
#pragma unroll
    for( int r = 0; r < H; ++r )
        t = cadd( t, a[r] );
    v[0] = t;
#pragma unroll
    for( int k = 1; k <= H; ++k )
    {
        double2 c = v0, s = make_double2( 0, 0 );
#pragma unroll
        for( int r = 1; r <= H; ++r )
        {
            const int m      = ( k * r ) % R;
            const double cr  = OddRoots<R>::c[( m <= H ? m : R - m ) - 1];
            const double sr  = m <= H ? OddRoots<R>::s[m - 1] : -OddRoots<R>::s[R - m - 1];
            c.x += cr * a[r - 1].x;
            c.y += cr * a[r - 1].y;
            s.x += sr * b[r - 1].x;
            s.y += sr * b[r - 1].y;
        }
        // forward: X[k] = c - i s, X[R-k] = c + i s
        const double2 lo = make_double2( c.x + s.y, c.y - s.x ), hi = make_double2( c.x - s.y, c.y + s.x );
        v[k]     = INV ? hi : lo;
        v[R - k] = INV ? lo : hi;
    }
}

template<int R, bool INV>
__device__ __forceinline__ void mix_dft( double2 * v );

// the multiple of b that is 1 mod a
constexpr int crt_unit( int a, int b )
{
    int e = b;
    while( e % a != 1 % a )
        e += b;
    return e;
}

// R = N1 N2 with coprime factors: no twiddles between the two (Good-Thomas)
template<int N1, int N2, bool INV>
__device__ __forceinline__ void dft_coprime( double2 * v )
{
    constexpr int R  = N1 * N2;
    constexpr int E1 = crt_unit( N1, N2 ), E2 = crt_unit( N2, N1 );
    double2 t[N2][N1];
#pragma unroll
    for( int n2 = 0; n2 < N2; ++n2 )
    {
#pragma unroll
        for( int n1 = 0; n1 < N1; ++n1 )
            t[n2][n1] = v[( N2 * n1 + N1 * n2 ) % R];
        mix_dft<N1, INV>( t[n2] );
    }
#pragma unroll
    for( int k1 = 0; k1 < N1; ++k1 )
    {
        double2 u[N2];
#pragma unroll
        for( int n2 = 0; n2 < N2; ++n2 )
            u[n2] = t[n2][k1];
        mix_dft<N2, INV>( u );
#pragma unroll
        for( int k2 = 0; k2 < N2; ++k2 )
        {
            // the output index that is k1 mod N1 and k2 mod N2
            v[( E1 * k1 + E2 * k2 ) % R] = u[k2];
        }
    }
}

// 9 = 3 x 3 with the twiddles w_9^(n2 k1) between the two
template<bool INV>
__device__ __forceinline__ void dft_9( double2 * v )
{
    double2 a[3] = { v[0], v[3], v[6] }, b[3] = { v[1], v[4], v[7] }, c[3] = { v[2], v[5], v[8] };
    dft_odd<3, INV>( a );
    dft_odd<3, INV>( b );
    dft_odd<3, INV>( c );
    const double sg  = INV ? 1.0 : -1.0;
    const double2 w1 = make_double2( 0.76604444311897803520, sg * 0.64278760968653932632 );
    const double2 w2 = make_double2( 0.17364817766693034885, sg * 0.98480775301220805937 );
    const double2 w4 = make_double2( -0.93969262078590838405, sg * 0.34202014332566873304 );
    double2 x[3] = { a[0], b[0], c[0] };
    double2 y[3] = { a[1], cmul( b[1], w1 ), cmul( c[1], w2 ) };
    double2 z[3] = { a[2], cmul( b[2], w2 ), cmul( c[2], w4 ) };
    dft_odd<3, INV>( x );
    dft_odd<3, INV>( y );
    dft_odd<3, INV>( z );
    v[0] = x[0], v[1] = y[0], v[2] = z[0];
    v[3] = x[1], v[4] = y[1], v[5] = z[1];
    v[6] = x[2], v[7] = y[2], v[8] = z[2];
}

// unnormalised DFT of R values in registers
template<int R, bool INV>
__device__ __forceinline__ void mix_dft( double2 * v )
{
    if constexpr( R == 1 )
        return;
    else if constexpr( R == 2 || R == 4 || R == 8 )
        dft_small<R, INV>( v );
    else if constexpr( R == 6 )
        dft_coprime<2, 3, INV>( v );
    else if constexpr( R == 9 )
        dft_9<INV>( v );
    else if constexpr( R == 10 )
        dft_coprime<2, 5, INV>( v );
    else if constexpr( R == 12 )
        dft_coprime<3, 4, INV>( v );
    else
        dft_odd<R, INV>( v );
}

// most butterflies of radix R a thread holds in an in-place stage (ten values, eight above radix 7)
template<int R>
struct MixPer
{
    static constexpr int PER = mix_per( R );
};

// The tile a block transforms: nl lines, LDS row stride lsr, m threads a line; a tile of more
// lines than the block has threads for is taken in groups of nc lines.
// TW_LDS: the twiddles are copied behind the tile, else they are read from the plan's table.
template<bool TW_LDS = true>
struct MixBlock
{
    int nl, lsr, nc, m;
    int lc, j0; // this thread's line in a group and its first butterfly
    double2 * lds;
    const double2 * tw;
    __device__ __forceinline__ MixBlock( const MixTile & T, const MixPlan & P, double2 * mem )
            : nl( T.nl ), lsr( T.lsr ), nc( T.nc ), m( T.m ), lds( mem ), tw( TW_LDS ? mem + P.n * T.lsr : P.tw )
    {
        j0 = (int)threadIdx.x / nc;
        lc = (int)threadIdx.x - j0 * nc;
        if constexpr( TW_LDS )
        {
            // settled by the barrier behind the first stage
            double2 * t = mem + P.n * T.lsr;
            for( int e = threadIdx.x; e < P.n_tw; e += blockDim.x )
                t[e] = P.tw[e];
        }
    }
    __device__ __forceinline__ double2 & at( int p, int l ) const
    {
        return lds[p * lsr + l];
    }
};

// stage s of a plan, through the scalar cache (the table does not change while a kernel runs)
__device__ __forceinline__ MixStage mix_stage( const MixPlan & P, int s )
{
    typedef const __attribute__( ( address_space( 4 ) ) ) MixStage * Table;
    const Table t = (Table)(uintptr_t)P.st + s;
    MixStage S;
    S.R         = t->R;
    S.Ns        = t->Ns;
    S.nbf       = t->nbf;
    S.tw        = t->tw;
    S.by_ns.inv = t->by_ns.inv;
    return S;
}

// A thread's first butterfly, opaque to the optimiser: the index arithmetic of a stage stays inside
// its radix's branch (hoisted out of the radix switch, the variants' indices spill registers).
template<typename BLK>
__device__ __forceinline__ int mix_j0( const BLK & T )
{
    int t = T.j0;
    asm volatile( "" : "+v"( t ) );
    return t;
}

// ... and the same for a uniform number
__device__ __forceinline__ int mix_opaque( int x )
{
    asm volatile( "" : "+s"( x ) );
    return x;
}

// first stage: inputs from ld( l, point ), outputs to st( l, position, value )
template<int R, bool INV, typename BLK, typename LD, typename ST>
__device__ __forceinline__ void mix_first( const MixStage & S, const BLK & T, LD ld, ST st )
{
    const int nbf = mix_opaque( S.nbf );
#pragma unroll 1
    for( int l = T.lc; l < T.nl; l += T.nc )
#pragma unroll 1
        for( int j = mix_j0( T ); j < nbf; j += T.m )
        {
            double2 u[R];
#pragma unroll
            for( int r = 0; r < R; ++r )
                u[r] = ld( l, j + r * nbf );
            mix_dft<R, INV>( u );
#pragma unroll
            for( int r = 0; r < R; ++r )
                st( l, j * R + r, u[r] );
        }
}

template<int R, bool INV, typename BLK>
__device__ __forceinline__ void mix_twiddle( const BLK & T, const MixStage & S, int jm, double2 * u )
{
    if( S.Ns == 1 )
        return;
    const double2 * tw = T.tw + S.tw + jm;
#pragma unroll
    for( int r = 1; r < R; ++r )
    {
        double2 w = tw[( r - 1 ) * S.Ns];
        if( INV )
            w.y = -w.y;
        u[r] = cmul( u[r], w );
    }
}

// a stage from LDS to LDS, in place; every thread of the block calls it; LDS is settled on return
template<int R, bool INV, typename BLK>
__device__ __forceinline__ void mix_mid( const MixStage & S, const BLK & T )
{
    if constexpr( R == 1 )
        return; // a line of one point
    constexpr int PER = MixPer<R>::PER;
    const int nbf     = mix_opaque( S.nbf ), Ns = mix_opaque( S.Ns );
#pragma unroll 1
    for( int l0 = 0; l0 < T.nl; l0 += T.nc )
    {
        const int j0 = mix_j0( T );
        const int l  = l0 + T.lc;
        double2 v[PER][R];
#pragma unroll
        for( int k = 0; k < PER; ++k )
        {
            const int j = j0 + k * T.m;
            if( j < nbf )
            {
#pragma unroll
                for( int r = 0; r < R; ++r )
                    v[k][r] = T.at( j + r * nbf, l );
            }
        }
        __syncthreads();
#pragma unroll
        for( int k = 0; k < PER; ++k )
        {
            const int j = j0 + k * T.m;
            if( j < nbf )
            {
                const int jm = j - mix_div( j, S.by_ns ) * Ns;
                mix_twiddle<R, INV>( T, S, jm, v[k] );
                mix_dft<R, INV>( v[k] );
                const int o = ( j - jm ) * R + jm;
#pragma unroll
                for( int r = 0; r < R; ++r )
                    T.at( o + r * Ns, l ) = v[k][r];
            }
        }
        __syncthreads();
    }
}

// last stage: inputs from LDS, output of point p of line l to st( l, p, value )
template<int R, bool INV, typename BLK, typename ST>
__device__ __forceinline__ void mix_last( const MixStage & S, const BLK & T, ST st )
{
    const int nbf = mix_opaque( S.nbf );
#pragma unroll 1
    for( int l = T.lc; l < T.nl; l += T.nc )
#pragma unroll 1
        for( int j = mix_j0( T ); j < nbf; j += T.m )
        {
            double2 u[R];
#pragma unroll
            for( int r = 0; r < R; ++r )
                u[r] = T.at( j + r * nbf, l );
            mix_twiddle<R, INV>( T, S, j, u );
            mix_dft<R, INV>( u );
#pragma unroll
            for( int r = 0; r < R; ++r )
                st( l, j + r * nbf, u[r] ); // Ns R = n: position j + r n / R
        }
}

// WIDE: the kernel also holds the radices 11 to 13, whose registers cost it occupancy (128 and
// spills instead of 92 to 114), for lengths with a factor 11 or 13
#define MIX_RADIX( R, call )                                                                                           \
    switch( R )                                                                                                        \
    {                                                                                                                  \
        case 1: call( 1 ); break;                                                                                      \
        case 2: call( 2 ); break;                                                                                      \
        case 3: call( 3 ); break;                                                                                      \
        case 4: call( 4 ); break;                                                                                      \
        case 5: call( 5 ); break;                                                                                      \
        case 6: call( 6 ); break;                                                                                      \
        case 7: call( 7 ); break;                                                                                      \
        case 8: call( 8 ); break;                                                                                      \
        case 9: call( 9 ); break;                                                                                      \
        case 10: call( 10 ); break;                                                                                    \
        default:                                                                                                       \
            if constexpr( WIDE )                                                                                       \
            {                                                                                                          \
                if( R == 11 )                                                                                          \
                    call( 11 );                                                                                        \
                else if( R == 12 )                                                                                     \
                    call( 12 );                                                                                        \
                else                                                                                                   \
                    call( 13 );                                                                                        \
            }                                                                                                          \
            break;                                                                                                     \
    }

template<bool INV, bool WIDE, typename BLK>
__device__ __forceinline__ void mix_mid_any( const MixPlan & P, const BLK & T, int s )
{
    const MixStage S = mix_stage( P, s );
#define MIX_CALL( R ) mix_mid<R, INV>( S, T )
    MIX_RADIX( S.R, MIX_CALL )
#undef MIX_CALL
}

// The transform of ld's inputs left in LDS in natural order (settled on return).
template<bool INV, bool WIDE, typename BLK, typename LD>
__device__ __forceinline__ void mix_fft_to_lds( const MixPlan & P, const BLK & T, LD ld )
{
    const MixStage S0 = mix_stage( P, 0 );
    auto put          = [&]( int l, int p, double2 v ) { T.at( p, l ) = v; };
#define MIX_CALL( R ) mix_first<R, INV>( S0, T, ld, put )
    MIX_RADIX( S0.R, MIX_CALL )
#undef MIX_CALL
    __syncthreads();
    for( int s = 1; s < P.ns; ++s )
        mix_mid_any<INV, WIDE>( P, T, s );
}

template<bool INV, bool WIDE, typename BLK, typename ST>
__device__ __forceinline__ void mix_last_any( const MixPlan & P, const BLK & T, ST st )
{
    const MixStage S = mix_stage( P, P.ns - 1 );
#define MIX_CALL( R ) mix_last<R, INV>( S, T, st )
    MIX_RADIX( S.R, MIX_CALL )
#undef MIX_CALL
}

// From ld's inputs to st's outputs.
template<bool INV, bool WIDE, typename BLK, typename LD, typename ST>
__device__ __forceinline__ void mix_fft( const MixPlan & P, const BLK & T, LD ld, ST st )
{
    const MixStage S0 = mix_stage( P, 0 );
    if( P.ns == 1 )
    {
#define MIX_CALL( R ) mix_first<R, INV>( S0, T, ld, st )
        MIX_RADIX( S0.R, MIX_CALL )
#undef MIX_CALL
        return;
    }
    auto put = [&]( int l, int p, double2 v ) { T.at( p, l ) = v; };
#define MIX_CALL( R ) mix_first<R, INV>( S0, T, ld, put )
    MIX_RADIX( S0.R, MIX_CALL )
#undef MIX_CALL
    __syncthreads();
    for( int s = 1; s < P.ns - 1; ++s )
        mix_mid_any<INV, WIDE>( P, T, s );
    mix_last_any<INV, WIDE>( P, T, st );
}

// From LDS (natural order, settled) to st's outputs.
template<bool INV, bool WIDE, typename BLK, typename ST>
__device__ __forceinline__ void mix_fft_from_lds( const MixPlan & P, const BLK & T, ST st )
{
    for( int s = 0; s < P.ns - 1; ++s )
        mix_mid_any<INV, WIDE>( P, T, s );
    mix_last_any<INV, WIDE>( P, T, st );
}

} // namespace spirit_hip
