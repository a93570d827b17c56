// Device helpers the passes of the dipolar FFT convolution share: the kernel spectrum, its
// product with the spin spectrum and the block order of the convolution pass.
#pragma once

#include "ddi.hpp"
#include "fft_small.hpp"

namespace spirit_hip
{

// ---------------------------------------------------------------------------
// kernel spectrum access and the symmetric 3x3 multiply (FFT.hpp:89-96 row order)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void dhat_load( const DdiDev & d, int kb, int ka, int kc, int b_inter, double2 * D )
{
    int kbs = kb, kcs = kc;
    bool mb = false, mc = false;
    if( d.sym_b && kb > d.Pb / 2 )
    {
        kbs = d.Pb - kb;
        mb  = true;
    }
    if( d.sym_c && kc > d.Pc / 2 )
    {
        kcs = d.Pc - kc;
        mc  = true;
    }
    const long long off = ( ( (long long)kbs * d.Ha + ka ) * d.KC + kcs ) * ( 6 * d.n_inter ) + 6 * b_inter;
#pragma unroll
    for( int q = 0; q < 6; ++q )
    {
        double2 v = d.dh_real ? make_double2( d.Dh_r[off + q], 0.0 ) : d.Dh[off + q];
        int sg    = ( mb ? d.sig_b[q] : 1 ) * ( mc ? d.sig_c[q] : 1 );
        if( sg < 0 )
        {
            v.x = -v.x;
            v.y = -v.y;
        }
        D[q] = v;
    }
}

// res_q = sum_p D_qp s_p, D symmetric (xx,xy,xz,yy,yz,zz)
__device__ __forceinline__ void sym3_mul( const double2 * D, const double2 * s, double2 * r )
{
    const int rows[3][3] = { { 0, 1, 2 }, { 1, 3, 4 }, { 2, 4, 5 } };
#pragma unroll
    for( int q = 0; q < 3; ++q )
    {
        const double2 d1 = D[rows[q][0]], d2 = D[rows[q][1]], d3 = D[rows[q][2]];
        r[q].x = d1.x * s[0].x + d2.x * s[1].x + d3.x * s[2].x - d1.y * s[0].y - d2.y * s[1].y - d3.y * s[2].y;
        r[q].y = d1.x * s[0].y + d2.x * s[1].y + d3.x * s[2].y + d1.y * s[0].x + d2.y * s[1].x + d3.y * s[2].x;
    }
}

// Hhat(b1) = sum_b2 Dhat(inter(b1,b2)) . Shat(b2) at one (kb, ka, kc); values in LDS at
// lds[line(arr) * ls + pos], arr = 3*basis + component.  ONE: the plan has one basis atom.
template<bool ONE = false, typename IDX>
__device__ __forceinline__ void conv_point( const DdiDev & d, int kb, int ka, int kc, double2 * lds, IDX idx )
{
    if( ( ONE || d.nb == 1 ) && d.dh_real )
    {
        // real spectrum: six values of the stored octant, the mirror's signs (dhat_load), and 18
        // real products instead of 36
        const bool mb   = d.sym_b && kb > d.Pb / 2, mc = d.sym_c && kc > d.Pc / 2;
        const int kbs   = mb ? d.Pb - kb : kb, kcs = mc ? d.Pc - kc : kc;
        const double2 * p
            = reinterpret_cast<const double2 *>( d.Dh_r + ( ( (long long)kbs * d.Ha + ka ) * d.KC + kcs ) * 6 );
        const double2 p0 = p[0], p1 = p[1], p2 = p[2];
        const double gb = mb ? -1.0 : 1.0, gc = mc ? -1.0 : 1.0;
        const double xx = p0.x, xy = gb * p0.y, xz = gc * p1.x, yy = p1.y, yz = gb * gc * p2.x, zz = p2.y;
        const double2 s0 = lds[idx( 0 )], s1 = lds[idx( 1 )], s2 = lds[idx( 2 )];
        lds[idx( 0 )] = make_double2( xx * s0.x + xy * s1.x + xz * s2.x, xx * s0.y + xy * s1.y + xz * s2.y );
        lds[idx( 1 )] = make_double2( xy * s0.x + yy * s1.x + yz * s2.x, xy * s0.y + yy * s1.y + yz * s2.y );
        lds[idx( 2 )] = make_double2( xz * s0.x + yz * s1.x + zz * s2.x, xz * s0.y + yz * s1.y + zz * s2.y );
        return;
    }
    if( ONE || d.nb == 1 )
    {
        double2 D[6], s[3], r[3];
        dhat_load( d, kb, ka, kc, 0, D );
#pragma unroll
        for( int q = 0; q < 3; ++q )
            s[q] = lds[idx( q )];
        sym3_mul( D, s, r );
#pragma unroll
        for( int q = 0; q < 3; ++q )
            lds[idx( q )] = r[q];
        return;
    }
    double2 S[MAX_BASIS][3];
    for( int b2 = 0; b2 < d.nb; ++b2 )
        for( int q = 0; q < 3; ++q )
            S[b2][q] = lds[idx( 3 * b2 + q )];
    for( int b1 = 0; b1 < d.nb; ++b1 )
    {
        double2 acc[3];
        for( int b2 = 0; b2 < d.nb; ++b2 )
        {
            double2 D[6], r[3];
            dhat_load( d, kb, ka, kc, d.inter[b1 + b2 * d.nb], D );
            sym3_mul( D, S[b2], r );
#pragma unroll
            for( int q = 0; q < 3; ++q )
                acc[q] = b2 == 0 ? r[q] : cadd( acc[q], r[q] );
        }
        for( int q = 0; q < 3; ++q )
            lds[idx( 3 * b1 + q )] = acc[q];
    }
}

// Logical block lb of a pass C launch (n_tiles column tiles per kb plane, Pb planes) to its
// (tile, kb).  With order_pairs: plane 0, then for 0 < p < Pb-p the tiles of the planes p and
// Pb-p interleaved (tile j of p, tile j of Pb-p, ...), then plane Pb/2 if Pb is even, so the
// second read of a stored spectrum tile (the two planes share it) follows the first by one
// block and hits in L2.  A bijection on [0, n_tiles * Pb).
__device__ __forceinline__ void pass_c_block( int lb, int n_tiles, int Pb, int order_pairs, int & tile, int & kb )
{
    tile = lb % n_tiles;
    kb   = lb / n_tiles;
    if( !order_pairs || lb < n_tiles )
        return;
    const int r     = lb - n_tiles;
    const int pairs = ( Pb - 1 ) / 2; // planes p and Pb-p with 0 < p < Pb-p
    if( r < 2 * n_tiles * pairs )
    {
        const int p = 1 + r / ( 2 * n_tiles );
        const int w = r % ( 2 * n_tiles );
        tile        = w >> 1;
        kb          = ( w & 1 ) ? Pb - p : p;
    }
    else
    {
        tile = r - 2 * n_tiles * pairs;
        kb   = Pb / 2;
    }
}

} // namespace spirit_hip
