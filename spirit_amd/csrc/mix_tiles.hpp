// Shapes of the mixed-radix transforms (fft_mix.hpp): the radices of a length, and the tile of lines
// a block transforms with the threads a line gets.  Plain C++, for the host.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <functional>
#include <stdexcept>
#include <string>
#include <vector>

namespace spirit_hip
{

constexpr int MAX_MIX_STAGES  = 5;    // enough for every length to 4096 with prime factors to 13
constexpr int MIX_MAX_THREADS = 1024; // of a block

// most butterflies of radix R a thread holds in an in-place stage
constexpr int mix_per( int R )
{
    return R >= 8 ? 1 : ( 10 + R - 1 ) / R;
}

// A tile of lines (MixBlock): nl lines in groups of nc, LDS row stride lsr, m threads a line.
struct MixTile
{
    int nl, lsr, nc, m;
};

// A length: its ns radices, the largest first, and the entries of its stage-twiddle table.
struct MixLen
{
    int n, ns, n_tw;
    int radix[MAX_MIX_STAGES];
};

// The radices of n (at most 10, or 13 with a factor 11 or 13): as few stages as possible, then the
// smallest largest radix (registers), then the smallest sum; the largest first, where half of a
// zero-padded line's inputs need no load.
inline MixLen mix_length( int n )
{
    std::vector<int> best, now;
    auto better = [&]( const std::vector<int> & a ) {
        if( best.empty() )
            return true;
        if( a.size() != best.size() )
            return a.size() < best.size();
        if( a[0] != best[0] )
            return a[0] < best[0];
        int sa = 0, sb = 0;
        for( size_t k = 0; k < a.size(); ++k )
            sa += a[k], sb += best[k];
        return sa < sb;
    };
    // radices in descending order
    std::function<void( int, int )> search = [&]( int m, int top ) {
        if( m == 1 )
        {
            if( better( now ) )
                best = now;
            return;
        }
        if( (int)now.size() == MAX_MIX_STAGES )
            return;
        for( int r = std::min( top, m ); r >= 2; --r )
            if( m % r == 0 )
            {
                now.push_back( r );
                search( m / r, r );
                now.pop_back();
            }
    };
    if( n == 1 )
        best = { 1 };
    else
        search( n, n % 11 == 0 || n % 13 == 0 ? 13 : 10 );
    if( best.empty() )
        throw std::runtime_error( "DDI FFT: no mixed-radix plan for length " + std::to_string( n ) );
    MixLen L{ n, (int)best.size(), 0, {} };
    std::copy( best.begin(), best.end(), L.radix );
    for( int s = 1, Ns = L.radix[0]; s < L.ns; Ns *= L.radix[s++] )
        L.n_tw += ( L.radix[s] - 1 ) * Ns;
    return L;
}

// bytes of FP64 complex values: a tile of rows of lsr values and, with tw_lds, the twiddles behind it
inline size_t mix_lds( const MixLen & L, int lsr, bool tw_lds = true )
{
    return 16 * ( (size_t)L.n * (size_t)lsr + (size_t)( tw_lds ? L.n_tw : 0 ) );
}

// fewest threads a line needs: what the in-place stages' registers hold (mix_per)
inline int mix_least_threads( const MixLen & L )
{
    int lo = 1;
    for( int s = 0; s < L.ns; ++s )
        lo = std::max( lo, ( L.n / L.radix[s] + mix_per( L.radix[s] ) - 1 ) / mix_per( L.radix[s] ) );
    return lo;
}

// The tile of nl lines and the threads a line gets: at least mix_least_threads, and of the counts up to
// a quarter of the line the one with the fewest idle lanes over the stages and wavefronts, weighed
// against the waves a CU then holds (sixteen at the kernels' registers).  All lines at once, or, unless
// whole, the largest divisor of nl whose threads fit a block.
inline MixTile mix_tile( const MixLen & L, int nl, int lsr, bool whole, size_t lds_max, bool tw_lds = true )
{
    const int blocks = std::max( 1, (int)( lds_max / mix_lds( L, lsr, tw_lds ) ) );
    const int lo     = mix_least_threads( L );
    MixTile best{ nl, lsr, whole ? nl : 1, lo };
    double best_score = -1;
    for( int m = lo; m <= std::max( lo, ( L.n + 3 ) / 4 ); ++m )
    {
        int nc = nl;
        while( !whole && nc > 1 && ( nc * m > MIX_MAX_THREADS || nl % nc != 0 ) )
            --nc;
        double rounds = 0;
        for( int s = 0; s < L.ns; ++s )
            rounds += ( L.n / L.radix[s] + m - 1 ) / m * L.radix[s];
        const int waves    = ( nc * m + 63 ) / 64;
        const double use   = (double)L.n * L.ns / ( rounds * m ) * ( nc * m ) / ( 64.0 * waves );
        const double score = use * std::sqrt( std::min( 1.0, blocks * waves / 16.0 ) );
        if( nc * m <= MIX_MAX_THREADS && score > best_score + 1e-9 )
            best_score = score, best.nc = nc, best.m = m;
    }
    return best;
}

// Lines of a tile (a power of two), of n_lines altogether, `arrays` lines in LDS for each; fewer than
// `least` only where LDS forces it.
inline int mix_lines( const MixLen & L, int arrays, long long n_lines, int want, int least, size_t lds_max,
                      bool tw_lds = true )
{
    int cw = want;
    while( cw > 1
           && ( mix_lds( L, arrays * cw, tw_lds ) > lds_max / ( cw > 8 ? 2 : 1 )
                || ( cw > least && ( n_lines + cw - 1 ) / cw < 192 ) ) )
        cw /= 2;
    return cw;
}

// The tile of a pass whose threads keep one line for the whole transform (A, A^-1, B, B^-1): no more
// lines than the block has threads for; nl = 0 where none fits.
inline MixTile mix_line_tile( const MixLen & L, long long n_lines, int want, int least, size_t lds_max )
{
    int cw = mix_lines( L, 1, n_lines, want, least, lds_max );
    while( cw > 1 && cw * mix_least_threads( L ) > MIX_MAX_THREADS )
        cw /= 2;
    if( mix_lds( L, cw ) > lds_max || cw * mix_least_threads( L ) > MIX_MAX_THREADS )
        return MixTile{ 0, 0, 0, 0 };
    return mix_tile( L, cw, cw, true, lds_max );
}

// Pass A: row pairs are contiguous whatever their number is: 4, fewer where that fills the chip, and 16
// of rows so short that 4 of them leave most of a wavefront idle (a Heun step of 1x512x512 spins takes
// 418 us instead of 517, of 5x100x60 90 / 103, of 13x100x60 140 / 150; from 28 points on within 2%).
inline MixTile mix_row_tile( const MixLen & L, long long n_lines, size_t lds_max )
{
    return mix_line_tile( L, n_lines, L.n <= 26 ? 16 : 4, 1, lds_max );
}

// Column tiles no wider than a row of the spectrum needs.
inline int mix_width( int want, int row )
{
    while( want / 2 >= row )
        want /= 2;
    return want;
}

// Pass B: a row piece of a column tile is 16 cw bytes, so tiles are 16 wide where two blocks then fit a
// CU's LDS, else 8, and narrower only where LDS forces it or fewer than 192 blocks would leave CUs
// idle (not below 4, 64 bytes): 14 us a pass against 18 and 22 at 16, 8, 4 columns of 300 points, 13
// against 16 and 22 at 8, 4, 2 of 1000.
inline MixTile mix_column_tile( const MixLen & L, long long n_rows, int row, size_t lds_max )
{
    return mix_line_tile( L, n_rows * row, mix_width( 16, row ), 4, lds_max );
}

// The tile of a pass that holds `arrays` lines of each of its cw columns (line = array * cw + column, taken
// in groups where the threads need it); t.nl = 0 where none fits.
struct MixArraysTile
{
    MixTile t;
    int cw;
    bool tw_lds;
};
inline MixArraysTile mix_arrays_tile( const MixLen & L, int arrays, long long n_cols, int want, int least,
                                      size_t lds_max, bool tw_lds )
{
    const int cw = mix_lines( L, arrays, n_cols, want, least, lds_max, tw_lds );
    // an odd row stride spreads column accesses over the banks
    int lsr = ( arrays * cw ) | 1;
    if( mix_lds( L, lsr, tw_lds ) > lds_max )
        lsr = arrays * cw;
    if( mix_lds( L, lsr, tw_lds ) > lds_max || mix_least_threads( L ) > MIX_MAX_THREADS )
        return MixArraysTile{ MixTile{ 0, 0, 0, 0 }, 0, tw_lds };
    return MixArraysTile{ mix_tile( L, arrays * cw, lsr, false, lds_max, tw_lds ), cw, tw_lds };
}

// Pass C of n_arrays fields on n_rows rows of `row` columns, or the one-plane convolution along b (one
// row); want: the widest tile.  A block holds all arrays of its columns, which is much work for one, so
// the tiles narrow further than pass B's where blocks are few: pass C's to two columns (a Heun step of
// 12x12x50 cells of eight atoms takes 247 us instead of 527 with four, of four atoms 123 / 187, of one
// 65 / 65, 7x9x250 of one 78 / 84; one column is within 5% of two), the one along b to one.
// Where one column of pass C leaves no room for the twiddles (1463 to 1706 points of two basis atoms, 410
// to 426 of eight) they stay in global memory; a lattice of one plane has the passes along b instead.
inline MixArraysTile mix_conv_tile( const MixLen & L, int n_arrays, long long n_rows, int row, bool along_b, int want,
                                    size_t lds_max )
{
    const int w           = mix_width( want, row );
    const MixArraysTile C = mix_arrays_tile( L, n_arrays, n_rows * row, w, along_b ? 1 : 2, lds_max, true );
    return C.t.nl > 0 || along_b ? C : mix_arrays_tile( L, n_arrays, n_rows * row, 1, 1, lds_max, false );
}

// The kernel spectrum's pass C: the six components of a pair of sublattices.
inline MixArraysTile mix_spectrum_tile( const MixLen & L, long long n_rows, int row, size_t lds_max )
{
    return mix_arrays_tile( L, 6, n_rows * row, mix_width( 16, row ), 1, lds_max, false );
}

} // namespace spirit_hip
