// The passes of the dipolar FFT convolution for lengths that are no power of two (and the
// convolution pass wherever the power-of-two kernels do not apply), and the kernel spectrum's set-up
// at every length, hand-written for gfx950 on the mixed-radix tile transform of fft_mix.hpp.
//
// Every pass moves its part of the spectrum once (the padded half neither read nor written) and
// is bound by that traffic: a block transforms a tile of lines held in LDS, its first stage reads
// global memory straight into registers and its last one writes straight from them.  Two real
// rows share one complex transform in passes A and A^-1.
//
// Measured on a 200x150x12 film (padded 400x300x24, 36 MB of spectrum, in the memory-side cache),
// us a launch, against the one-row, one-stage-at-a-time LDS kernels these replaced: A 13 (47),
// B 14 (40), C 31 (74), B^-1 14 (40), A^-1 13 (54); reading and writing their data once takes
// 5, 10, 17, 10 and 5 at 5.4 TB/s.  What is left in A, B and their inverses is the chain load,
// three stages with two barriers each, store, of too few waves to overlap (11 to 15 a CU, waiting 51
// to 60% of their time; LDS is busy for 13 to 19%); pass C issues vector instructions half of its time.
#include "ddi_device.hpp"
#include "fft_mix.hpp"

namespace spirit_hip
{

// Passes A, A^-1, B and B^-1 derive their addresses from the thread's line once: their tiles have a
// thread for every line (T.nc == T.nl, mix_line_tile).

// Pass A: row pairs (b0 = 2 bp, b0 + 1) of one component and plane, zero-padded.
template<bool WIDE>
__global__ void __launch_bounds__( 1024 )
    k_mix_a_fwd( DdiDev d, MixPlan P, MixTile tile, const double * __restrict__ s, int nos )
{
    extern __shared__ double2 lds[];
    const MixBlock<> T( tile, P, lds );
    const int N         = P.n;
    const int cw        = T.nl;
    const int l         = T.lc; // this thread's line
    const int npairs    = ( d.Nb + 1 ) / 2;
    const int n_lines   = 3 * d.nb * npairs * d.Nc;
    const int blk       = ( d.rev & DDI_REV_A_FWD ) ? gridDim.x - 1 - blockIdx.x : blockIdx.x;
    const int line      = blk * cw + l;
    const bool act      = line < n_lines;
    const int rest      = line / npairs;
    const int b0        = 2 * ( line - rest * npairs );
    const int arr       = rest / d.Nc;
    const int c         = rest - arr * d.Nc;
    const bool has1     = act && b0 + 1 < d.Nb;
    const int ib        = arr / 3;
    const int q         = arr - 3 * ib;
    const double mu     = act ? d.mu[ib] : 0.0;
    const double * row0 = s + (long long)q * nos + ib + (long long)d.nb * d.Na * ( b0 + (long long)d.Nb * c );
    const double * row1 = row0 + (long long)d.nb * d.Na;
    mix_fft_to_lds<false, WIDE>( P, T, [&]( int, int a ) {
        double2 v = make_double2( 0, 0 );
        if( act && a < d.Na )
        {
            v.x = row0[(long long)d.nb * a] * mu;
            if( has1 )
                v.y = row1[(long long)d.nb * a] * mu;
        }
        return v;
    } );
    if( !act )
        return;
    // Z = X1 + i X2 of two real rows: X1 = (Z + conj Z[-k]) / 2, X2 = (Z - conj Z[-k]) / (2i)
    double2 * out0 = d.X + ( ( (long long)arr * d.Nc + c ) * d.Pb + b0 ) * d.Hs;
    double2 * out1 = out0 + d.Hs;
    for( int k = T.j0; k < d.Ha; k += T.m )
    {
        const double2 z = T.at( k, l ), m = T.at( k == 0 ? 0 : N - k, l );
        out0[k] = make_double2( 0.5 * ( z.x + m.x ), 0.5 * ( z.y - m.y ) );
        if( has1 )
            out1[k] = make_double2( 0.5 * ( z.y + m.y ), -0.5 * ( z.x - m.x ) );
    }
}

// Pass A^-1: Z = X1 + i X2 from the stored halves of two Hermitian rows, h = mu res / M.
template<bool WIDE>
__global__ void __launch_bounds__( 1024 )
    k_mix_a_inv( DdiDev d, MixPlan P, MixTile tile, double * __restrict__ h, int nos )
{
    extern __shared__ double2 lds[];
    const MixBlock<> T( tile, P, lds );
    const int N          = P.n;
    const int cw         = T.nl;
    const int l          = T.lc;
    const int npairs     = ( d.Nb + 1 ) / 2;
    const int n_lines    = 3 * d.nb * npairs * d.Nc;
    const int blk        = ( d.rev & DDI_REV_A_INV ) ? gridDim.x - 1 - blockIdx.x : blockIdx.x;
    const int line       = blk * cw + l;
    const bool act       = line < n_lines;
    const int rest       = line / npairs;
    const int b0         = 2 * ( line - rest * npairs );
    const int arr        = rest / d.Nc;
    const int c          = rest - arr * d.Nc;
    const bool has1      = act && b0 + 1 < d.Nb;
    const int ib         = arr / 3;
    const int q          = arr - 3 * ib;
    const double mu      = act ? d.mu[ib] : 0.0;
    const double2 * row0 = d.X + ( ( (long long)arr * d.Nc + c ) * d.Pb + b0 ) * d.Hs;
    const double2 * row1 = row0 + d.Hs;
    double * h0          = h + (long long)q * nos + ib + (long long)d.nb * d.Na * ( b0 + (long long)d.Nb * c );
    double * h1          = h0 + (long long)d.nb * d.Na;
    mix_fft<true, WIDE>(
        P, T,
        [&]( int, int k ) {
            const bool half = k < d.Ha;
            const int kk    = half ? k : N - k;
            double2 x1 = make_double2( 0, 0 ), x2 = make_double2( 0, 0 );
            if( act )
                x1 = row0[kk];
            if( has1 )
                x2 = row1[kk];
            if( !half )
                x1.y = -x1.y, x2.y = -x2.y;
            return make_double2( x1.x - x2.y, x1.y + x2.x );
        },
        [&]( int, int a, double2 v ) {
            if( act && a < d.Na )
            {
                h0[(long long)d.nb * a] = mu * v.x / d.M;
                if( has1 )
                    h1[(long long)d.nb * a] = mu * v.y / d.M;
            }
        } );
}

// Pass B: columns along b of one (component, plane) slab, inputs b < b_in, outputs b < b_out.
template<bool INV, bool WIDE>
__global__ void __launch_bounds__( 1024 )
    k_mix_b( DdiDev d, MixPlan P, MixTile tile, double2 * __restrict__ X, int n_tiles, int b_in, int b_out )
{
    extern __shared__ double2 lds[];
    const MixBlock<> T( tile, P, lds );
    const int cw   = T.nl;
    const int l    = T.lc;
    const int bid  = ( d.rev & ( INV ? DDI_REV_B_INV : DDI_REV_B_FWD ) ) ? gridDim.x - 1 - blockIdx.x : blockIdx.x;
    const int slab = bid / n_tiles;
    const int ka   = ( bid - slab * n_tiles ) * cw + l;
    const bool col = ka < d.Ha;
    double2 * p    = X + (long long)slab * P.n * d.Hs + ka;
    mix_fft<INV, WIDE>(
        P, T,
        [&]( int, int b ) { return col && b < b_in ? p[(long long)b * d.Hs] : make_double2( 0, 0 ); },
        [&]( int, int b, double2 v ) {
            if( col && b < b_out )
                p[(long long)b * d.Hs] = v;
        } );
}

// The convolution along one axis: forward transform of all 3 nb arrays of cw columns (ka), the
// product with the kernel spectrum, inverse transform, the first n_in points kept.
// ALONG_B = false: pass C, the axis is c, one kb plane a block (planes kb and Pb-kb interleaved
// with order_pairs).  ALONG_B = true: a lattice of one plane has nothing to transform along c, so
// passes B, C and B^-1 are this one kernel along b.  ONE: one basis atom (the product over pairs of
// basis atoms indexes a private array, which costs scratch memory).  TW_LDS: MixBlock's.
template<bool ALONG_B, bool WIDE, bool ONE, bool TW_LDS = true>
__global__ void __launch_bounds__( 1024 )
    k_mix_conv( DdiDev d, MixPlan P, MixTile mt, double2 * __restrict__ X, int cw, MixDiv by_cw, MixDiv by_n,
                int n_tiles, int order_pairs )
{
    extern __shared__ double2 lds[];
    const MixBlock<TW_LDS> T( mt, P, lds );
    // XCD-contiguous block order: neighbouring column tiles share cache lines of a row
    const int nblk = gridDim.x;
    const int full = ( nblk / 8 ) * 8;
    int lb         = blockIdx.x;
    if( lb < full )
        lb = ( lb % 8 ) * ( full / 8 ) + lb / 8;
    int tile = lb, kb = 0;
    if( !ALONG_B )
        pass_c_block( lb, n_tiles, d.Pb, order_pairs, tile, kb );
    const int ka0         = tile * cw;
    const int nk          = min( cw, d.Ha - ka0 );
    const long long plane = (long long)d.Pb * d.Hs;
    const int n_in        = ALONG_B ? d.Nb : d.Nc;
    double2 * base        = ALONG_B ? X + ka0 : X + (long long)kb * d.Hs + ka0;
    const long long es    = ALONG_B ? d.Hs : plane;                   // one point further along the axis
    const long long as    = ALONG_B ? plane : plane * (long long)d.Nc; // one array further
    mix_fft_to_lds<false, WIDE>( P, T, [&]( int l, int p ) {
        const int arr = mix_div( l, by_cw ), col = l - arr * cw;
        return col < nk && p < n_in ? base[arr * as + p * es + col] : make_double2( 0, 0 );
    } );
    // one spectrum point a thread: along c the points of a column are contiguous in the stored
    // kernel spectrum, along b those of a row
    for( int e = threadIdx.x; e < cw * P.n; e += blockDim.x )
    {
        const int hi = mix_div( e, ALONG_B ? by_cw : by_n );
        const int lo = e - hi * ( ALONG_B ? cw : P.n );
        const int col = ALONG_B ? lo : hi, p = ALONG_B ? hi : lo;
        if( col < nk )
            conv_point<ONE>( d, ALONG_B ? p : kb, ka0 + col, ALONG_B ? 0 : p, lds,
                        [&]( int arr ) { return p * T.lsr + arr * cw + col; } );
    }
    __syncthreads();
    mix_fft_from_lds<true, WIDE>( P, T, [&]( int l, int p, double2 v ) {
        const int arr = mix_div( l, by_cw ), col = l - arr * cw;
        if( col < nk && p < n_in )
            base[arr * as + p * es + col] = v;
    } );
}

// ---------------------------------------------------------------------------
// the kernel spectrum (set-up)
// ---------------------------------------------------------------------------
// Rows along a: one real row a line, its half spectrum to a row of stride Hs.
template<bool WIDE>
__global__ void __launch_bounds__( 1024 )
    k_mix_rows( MixPlan P, MixTile tile, const double * __restrict__ src, double2 * __restrict__ out, long long n_rows,
                int Ha, int Hs )
{
    extern __shared__ double2 lds[];
    const MixBlock<> T( tile, P, lds );
    const long long row = (long long)blockIdx.x * T.nl + T.lc;
    const bool act      = row < n_rows;
    const double * in   = src + row * P.n;
    mix_fft_to_lds<false, WIDE>( P, T, [&]( int, int a ) { return make_double2( act ? in[a] : 0.0, 0.0 ); } );
    if( act )
        for( int k = T.j0; k < Ha; k += T.m )
            out[row * Hs + k] = T.at( k, T.lc );
}

// Columns along c of the six components of a pair of sublattices, all Pc planes, stored as
// Dfull[kb][ka][kc][6 * pair + component].
template<bool WIDE>
__global__ void __launch_bounds__( 1024 )
    k_mix_c_spectrum( DdiDev d, MixPlan P, MixTile mt, const double2 * __restrict__ X, double2 * __restrict__ Dfull, int cw,
                      MixDiv by_cw, int n_tiles )
{
    extern __shared__ double2 lds[];
    const MixBlock<false> T( mt, P, lds );
    const int rest        = blockIdx.x / n_tiles;
    const int ka0         = ( blockIdx.x - rest * n_tiles ) * cw;
    const int pair        = rest / d.Pb;
    const int kb          = rest - pair * d.Pb;
    const int nk          = min( cw, d.Ha - ka0 );
    const long long plane = (long long)d.Pb * d.Hs;
    const double2 * base  = X + 6LL * pair * P.n * plane + (long long)kb * d.Hs + ka0;
    mix_fft_to_lds<false, WIDE>( P, T, [&]( int l, int c ) {
        const int q = mix_div( l, by_cw ), col = l - q * cw;
        return col < nk ? base[( (long long)q * P.n + c ) * plane + col] : make_double2( 0, 0 );
    } );
    double2 * out = Dfull + ( (long long)kb * d.Ha + ka0 ) * P.n * ( 6 * d.n_inter ) + 6 * pair;
    for( int e = threadIdx.x; e < 6 * nk * P.n; e += blockDim.x )
    {
        const int at = e / 6, q = e - 6 * at;
        const int col = at / P.n, kc = at - col * P.n;
        out[(long long)at * ( 6 * d.n_inter ) + q] = T.at( kc, q * cw + col );
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static bool mix_wide( const DdiDev & d, int axis )
{
    return d.mix->len[axis].radix[0] > 10; // the largest radix is the first
}

static MixTile mix_a_tile( const DdiDev & d )
{
    return mix_row_tile( d.mix->len[0], 3LL * d.nb * ( ( d.Nb + 1 ) / 2 ) * d.Nc, d.lds_max );
}

static MixTile mix_b_tile( const DdiDev & d )
{
    return mix_column_tile( d.mix->len[1], 3LL * d.nb * d.Nc, d.Ha, d.lds_max );
}

bool mix_a_ok( const DdiDev & d )
{
    return mix_a_tile( d ).nl > 0;
}

bool mix_b_ok( const DdiDev & d )
{
    return mix_b_tile( d ).nl > 0;
}

static MixArraysTile mix_c_tile( const DdiDev & d, bool along_b, int want )
{
    return along_b ? mix_conv_tile( d.mix->len[1], 3 * d.nb, 1, d.Ha, true, want, d.lds_max )
                   : mix_conv_tile( d.mix->len[2], 3 * d.nb, d.Pb, d.Ha, false, want, d.lds_max );
}

bool mix_conv_ok( const DdiDev & d, bool along_b )
{
    return mix_c_tile( d, along_b, MIX_WIDEST ).t.nl > 0;
}

int mix_conv_width( const DdiDev & d )
{
    return mix_c_tile( d, false, MIX_WIDEST ).cw;
}

void mix_launch_a_fwd( const DdiDev & d, const double * s, int nos, hipStream_t st )
{
    const MixTile T       = mix_a_tile( d );
    const long long lines = 3LL * d.nb * ( ( d.Nb + 1 ) / 2 ) * d.Nc;
    const auto k          = mix_wide( d, 0 ) ? k_mix_a_fwd<true> : k_mix_a_fwd<false>;
    hipLaunchKernelGGL( k, dim3( (unsigned)( ( lines + T.nl - 1 ) / T.nl ) ), dim3( T.nc * T.m ),
                        mix_lds( d.mix->len[0], T.lsr ), st, d, d.mix->plan[0], T, s, nos );
}

void mix_launch_a_inv( const DdiDev & d, double * h, int nos, hipStream_t st )
{
    const MixTile T       = mix_a_tile( d );
    const long long lines = 3LL * d.nb * ( ( d.Nb + 1 ) / 2 ) * d.Nc;
    const auto k          = mix_wide( d, 0 ) ? k_mix_a_inv<true> : k_mix_a_inv<false>;
    hipLaunchKernelGGL( k, dim3( (unsigned)( ( lines + T.nl - 1 ) / T.nl ) ), dim3( T.nc * T.m ),
                        mix_lds( d.mix->len[0], T.lsr ), st, d, d.mix->plan[0], T, h, nos );
}

void mix_launch_b( const DdiDev & d, bool inverse, hipStream_t st )
{
    const MixTile T = mix_b_tile( d );
    const int tiles = ( d.Ha + T.nl - 1 ) / T.nl;
    const dim3 g( (unsigned)( (long long)tiles * d.Nc * 3 * d.nb ) ), b( T.nc * T.m );
    const bool w = mix_wide( d, 1 );
    const auto k = inverse ? ( w ? k_mix_b<true, true> : k_mix_b<true, false> )
                           : ( w ? k_mix_b<false, true> : k_mix_b<false, false> );
    hipLaunchKernelGGL( k, g, b, mix_lds( d.mix->len[1], T.lsr ), st, d, d.mix->plan[1], T, d.X, tiles,
                        inverse ? d.Pb : d.Nb, inverse ? d.Nb : d.Pb );
}

void mix_launch_conv( const DdiDev & d, bool along_b, int want, hipStream_t st )
{
    const int axis        = along_b ? 1 : 2;
    const MixPlan & P     = d.mix->plan[axis];
    const MixArraysTile C = mix_c_tile( d, along_b, want );
    const int tiles       = ( d.Ha + C.cw - 1 ) / C.cw;
    const MixDiv by_cw{ 1.0f / (float)C.cw }, by_n{ 1.0f / (float)P.n };
    const bool w = mix_wide( d, axis ), one = d.nb == 1;
    const auto k = along_b     ? ( w     ? k_mix_conv<true, true, false>
                                   : one ? k_mix_conv<true, false, true>
                                         : k_mix_conv<true, false, false> )
                   : !C.tw_lds ? k_mix_conv<false, true, false, false>
                               : ( w     ? k_mix_conv<false, true, false>
                                   : one ? k_mix_conv<false, false, true>
                                         : k_mix_conv<false, false, false> );
    hipLaunchKernelGGL( k, dim3( (unsigned)( (long long)tiles * ( along_b ? 1 : d.Pb ) ) ), dim3( C.t.nc * C.t.m ),
                        mix_lds( d.mix->len[axis], C.t.lsr, C.tw_lds ), st, d, P, C.t, d.X, C.cw, by_cw, by_n, tiles,
                        !along_b && d.sym_b ? 1 : 0 );
}

static MixArraysTile mix_c_spectrum_tile( const DdiDev & d )
{
    return mix_spectrum_tile( d.mix->len[2], (long long)d.Pb * d.n_inter, d.Ha, d.lds_max );
}

bool mix_spectrum_ok( const DdiDev & d )
{
    const long long n_slabs = 6LL * d.n_inter * d.Pc;
    return mix_row_tile( d.mix->len[0], n_slabs * d.Pb, d.lds_max ).nl > 0
           && mix_column_tile( d.mix->len[1], n_slabs, d.Ha, d.lds_max ).nl > 0 && mix_c_spectrum_tile( d ).t.nl > 0;
}

void mix_launch_spectrum( const DdiDev & d, const double * D, double2 * work, double2 * Dfull, hipStream_t st )
{
    const MixLen * L        = d.mix->len;
    const long long n_slabs = 6LL * d.n_inter * d.Pc;
    {
        const long long n_rows = n_slabs * d.Pb;
        const MixTile T        = mix_row_tile( L[0], n_rows, d.lds_max );
        const auto k           = mix_wide( d, 0 ) ? k_mix_rows<true> : k_mix_rows<false>;
        hipLaunchKernelGGL( k, dim3( (unsigned)( ( n_rows + T.nl - 1 ) / T.nl ) ), dim3( T.nc * T.m ),
                            mix_lds( L[0], T.lsr ), st, d.mix->plan[0], T, D, work, n_rows, d.Ha, d.Hs );
    }
    {
        const MixTile T = mix_column_tile( L[1], n_slabs, d.Ha, d.lds_max );
        const int tiles = ( d.Ha + T.nl - 1 ) / T.nl;
        const auto k    = mix_wide( d, 1 ) ? k_mix_b<false, true> : k_mix_b<false, false>;
        hipLaunchKernelGGL( k, dim3( (unsigned)( n_slabs * tiles ) ), dim3( T.nc * T.m ), mix_lds( L[1], T.lsr ), st, d,
                            d.mix->plan[1], T, work, tiles, d.Pb, d.Pb );
    }
    {
        const MixArraysTile C = mix_c_spectrum_tile( d );
        const int tiles       = ( d.Ha + C.cw - 1 ) / C.cw;
        const auto k          = mix_wide( d, 2 ) ? k_mix_c_spectrum<true> : k_mix_c_spectrum<false>;
        hipLaunchKernelGGL( k, dim3( (unsigned)( (long long)tiles * d.Pb * d.n_inter ) ), dim3( C.t.nc * C.t.m ),
                            mix_lds( L[2], C.t.lsr, false ), st, d, d.mix->plan[2], C.t, work, Dfull, C.cw,
                            MixDiv{ 1.0f / (float)C.cw }, tiles );
    }
}

} // namespace spirit_hip
