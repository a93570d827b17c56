"""The tiles of the mixed-radix dipolar passes over every accepted length and line count, from the host
header that the launches take them from: every line of a launch belongs to a thread, the threads of a
line hold its in-place stages, and the tile fits a block's threads and LDS.  No GPU is used."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SWEEP = r"""
#include "mix_tiles.hpp"
#include <cstdio>
#include <vector>
using namespace spirit_hip;

static const size_t LDS = 160 * 1024;
static int bad = 0, tiles = 0;

static bool smooth( int n )
{
    for( int p : { 2, 3, 5, 7, 11, 13 } )
        while( n % p == 0 )
            n /= p;
    return n == 1;
}

static void fail( const char * what, const MixLen & L, long long lines, const MixTile & T )
{
    if( ++bad < 40 )
        std::printf( "%s: n %d, %lld lines, tile nl %d lsr %d nc %d m %d\n", what, L.n, lines, T.nl, T.lsr, T.nc, T.m );
}

// what every kernel of the transform relies on
static void common( const char * pass, const MixLen & L, long long lines, const MixTile & T )
{
    ++tiles;
    bool ok = T.nl >= 1 && T.nc >= 1 && T.nl % T.nc == 0 && T.m >= 1 && T.nc * T.m <= MIX_MAX_THREADS && T.lsr >= T.nl;
    int n = 1;
    for( int s = 0; s < L.ns; n *= L.radix[s++] )
        // stages between the first and the last run in place, held in registers
        ok = ok && ( L.ns == 1 || (long long)T.m * mix_per( L.radix[s] ) >= L.n / L.radix[s] );
    if( !ok || n != L.n )
        fail( pass, L, lines, T );
}

static void arrays( const char * pass, const MixLen & L, long long cols, const MixArraysTile & C, int n )
{
    if( C.t.nl == 0 )
        return; // no tile fits: the plan is refused
    common( pass, L, cols, C.t );
    if( C.t.nl != n * C.cw || mix_lds( L, C.t.lsr, C.tw_lds ) > LDS )
        fail( pass, L, cols, C.t );
}

int main()
{
    std::vector<long long> counts;
    for( long long c = 1; c < 3000; c += 1 + c / 40 )
        counts.push_back( c );
    for( long long c = 3000; c < 5000000; c *= 3 )
        counts.push_back( c );
    for( int n = 1; n <= 4096; ++n )
    {
        if( !smooth( n ) )
            continue;
        const MixLen L = mix_length( n );
        int last_a = -1, last_b = -1;
        for( long long c : counts )
        {
            const int ca = mix_lines( L, 1, c, 16, 1, LDS ) + 100 * mix_lines( L, 1, c, 4, 1, LDS );
            const int cb = mix_lines( L, 1, c, 16, 4, LDS );
            if( ca != last_a )
            {
                // passes A and A^-1: a thread keeps the line (row pair) threadIdx mod nc
                const MixTile T = mix_row_tile( L, c, LDS );
                common( "rows", L, c, T );
                if( T.nc != T.nl || mix_lds( L, T.lsr ) > LDS )
                    fail( "rows: lines without a thread", L, c, T );
                last_a = ca;
            }
            if( cb != last_b )
            {
                // passes B and B^-1: the same for the columns
                for( int row : { 1, 2, 3, 5, 9, 201 } )
                {
                    const MixTile T = mix_column_tile( L, ( c + row - 1 ) / row, row, LDS );
                    common( "columns", L, c, T );
                    if( T.nc != T.nl || mix_lds( L, T.lsr ) > LDS || T.nl >= 2 * row )
                        fail( "columns: lines without a thread", L, c, T );
                }
                last_b = cb;
            }
            if( c > 3000 || c % 7 != 1 )
                continue;
            // passes that hold several arrays of a column: the convolution and the kernel spectrum
            for( int nb = 1; nb <= 8; ++nb )
                for( int along_b = 0; along_b < 2; ++along_b )
                    for( int want = 16; want >= 1; want /= 2 )
                        arrays( along_b ? "convolution along b" : "convolution along c", L, c,
                                mix_conv_tile( L, 3 * nb, along_b ? 1 : ( c + 200 ) / 201, along_b ? (int)c : 201,
                                               along_b, want, LDS ), 3 * nb );
            arrays( "kernel spectrum", L, c, mix_spectrum_tile( L, ( c + 2 ) / 3, 3, LDS ), 6 );
        }
    }
    std::printf( "%d tiles, %d bad\n", tiles, bad );
    return bad ? 1 : 0;
}
"""


def _compile(tmp_path, source, name):
    cxx = shutil.which("g++") or shutil.which("c++") or "/opt/rocm/bin/hipcc"
    src, exe = str(tmp_path / (name + ".cpp")), str(tmp_path / name)
    with open(src, "w") as f:
        f.write(source)
    subprocess.run([cxx, "-std=c++17", "-O1", "-I", os.path.join(ROOT, "spirit_amd", "csrc"), src, "-o", exe], check=True)
    return exe


# which (basis atoms, points along c) have a pass C: three lines of each atom, one value of padding a
# line, in a block's LDS, and the same for the kernel spectrum's six lines
LIMITS = r"""
#include "mix_tiles.hpp"
#include <cstdio>
#include <cstdlib>
using namespace spirit_hip;
int main()
{
    int n, nb;
    while( std::scanf( "%d %d", &nb, &n ) == 2 )
        std::printf( "%d %d %d %d\n", nb, n, mix_conv_tile( mix_length( n ), 3 * nb, 5, 201, false, 16, 160 * 1024 ).t.nl > 0,
                     mix_spectrum_tile( mix_length( n ), 5, 201, 160 * 1024 ).t.nl > 0 );
}
"""


def test_lengths_along_c_that_fit_without_their_twiddles(tmp_path):
    smooth = []
    for n in range(1, 4097):
        m = n
        for p in (2, 3, 5, 7, 11, 13):
            while m % p == 0:
                m //= p
        if m == 1:
            smooth.append(n)
    exe = _compile(tmp_path, LIMITS, "limits")
    asked = [(nb, n) for nb in range(1, 9) for n in smooth]
    out = subprocess.run([exe], input="\n".join("%d %d" % a for a in asked), capture_output=True, text=True, check=True)
    rows = [tuple(map(int, l.split())) for l in out.stdout.splitlines()]
    assert len(rows) == len(asked)
    for nb, n, conv, spectrum in rows:
        # 10240 complex values fit; the row padding of the lines is given up before the length
        assert conv == (3 * nb * n <= 10240), (nb, n)
        assert spectrum == (6 * n <= 10240), (nb, n)


def test_every_line_of_every_tile_has_a_thread(tmp_path):
    r = subprocess.run([_compile(tmp_path, SWEEP, "sweep")], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split()[0 if r.stdout[0].isdigit() else -4]) > 1000
