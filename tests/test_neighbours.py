"""The two neighbour lookups of the device code, compiled for the host: the one from a pair's fixed index
offset against the one from the cell's coordinates, over lattices of one to five cells an axis, every
combination of open and periodic axes, one and two basis atoms and translations up to and beyond the
lattice.  No GPU is used."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "neighbours.hpp"
#include <cstdio>
using namespace spirit_hip;
int main()
{
    long n = 0, bad = 0;
    const int sizes[] = { 1, 2, 3, 5 };
    for( int Na : sizes )
        for( int Nb : sizes )
            for( int Nc : { 1, 2, 4 } )
                for( int nb : { 1, 2 } )
                    for( int bc = 0; bc < 8; ++bc )
                        for( int da = -6; da <= 6; ++da )
                            for( int db = -6; db <= 6; ++db )
                                for( int dc = -5; dc <= 5; ++dc )
                                {
                                    HamDev H{};
                                    H.Na = Na, H.Nb = Nb, H.Nc = Nc, H.nb = nb;
                                    H.bc[0] = bc & 1, H.bc[1] = ( bc >> 1 ) & 1, H.bc[2] = bc >> 2;
                                    PairDev p{};
                                    p.i = ( da + 6 ) % nb, p.j = ( db + 6 ) % nb, p.da = da, p.db = db, p.dc = dc;
                                    p.delta = p.j - p.i + nb * ( da + Na * ( db + Nb * dc ) );
                                    for( int c = 0; c < Nc; ++c )
                                        for( int b = 0; b < Nb; ++b )
                                            for( int a = 0; a < Na; ++a, ++n )
                                            {
                                                const int i = p.i + nb * ( a + Na * ( b + Nb * c ) );
                                                bad += pair_neighbour( H, a, b, c, p )
                                                       != pair_neighbour_delta( H, i, a, b, c, p );
                                            }
                                }
    std::printf( "%ld sites, %ld bad\n", n, bad );
    return bad != 0;
}
"""


def test_neighbour_by_offset_is_the_neighbour_by_coordinates(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    src, exe = str(tmp_path / "neighbours.cpp"), str(tmp_path / "neighbours")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run([cxx, "-std=c++17", "-O2", "-w", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"), "-I",
                    os.path.join(ROOT, "spirit_amd", "csrc"), src, "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split()[0]) > 10 ** 7
