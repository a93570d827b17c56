"""The thermal draw's logarithm of a uniform number, compiled for the host, against the 80-bit logarithm: all
53 binades of the multiples of 2^-53 in (0, 1] with their ends, both sides of sqrt(1/2), 1 and its
neighbours, the smallest ones all; with products contracted into sums and without, and with reciprocals
off by as much as the device's may be.  Bound: the 1.1 units in the last place that the code states (half
a unit of the last sum, the rest from the correction's roundings).  No GPU is used."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "log_uniform.hpp"
#include <algorithm>
#include <cstdint>
#include <cstdio>
using namespace spirit_hip;

static double worst = 0, worst_u = 0, off;
static long count = 0;

static void check( uint64_t n )
{
    const uint64_t one = 1ull << 53;
    if( n < 1 || n > one )
        return;
    const double u   = (double)n / (double)one;
    const double got = log_uniform( u, []( double d ) { return 1.0 / d * ( 1.0 + off ); } );
    const long double want = logl( (long double)u );
    ++count;
    if( n == one )
    {
        if( got != 0.0 || std::signbit( -2.0 * got ) != std::signbit( -0.0 ) )
            worst = 1e30, worst_u = u;
        return;
    }
    int e;
    (void)frexpl( want, &e );
    const double ulps = (double)( std::fabs( (long double)got - want ) / ldexpl( 1.0L, e - 53 ) );
    if( !( ulps <= worst ) )
        worst = ulps, worst_u = u;
    if( !( got < 0.0 ) )
        worst = 1e30, worst_u = u;
}

int main()
{
    uint64_t x = 88172645463325252ull;
    for( double o : { 0.0, 0x1p-23, -0x1p-23 } )
    {
        off = o;
        for( uint64_t n = 1; n <= 5000; ++n )
            check( n ), check( ( 1ull << 53 ) + 1 - n );
        for( int b = 0; b <= 53; ++b )
        {
            const uint64_t lo   = 1ull << b;
            const uint64_t root = (uint64_t)( 0.70710678118654752 * 2.0 * (double)lo );
            for( uint64_t d = 0; d < 200; ++d )
                check( lo + d ), check( lo - d ), check( root + d ), check( root - d );
            for( int k = 0; k < 40000; ++k )
            {
                x ^= x << 13, x ^= x >> 7, x ^= x << 17;
                check( lo + ( x & ( lo - 1 ) ) );
            }
        }
    }
    std::printf( "%ld numbers, worst %.4f ulp at %a\n", count, worst, worst_u );
    return worst <= 1.1 ? 0 : 1;
}
"""


@pytest.mark.parametrize("contract", ["off", "fast"])
def test_log_of_a_uniform(tmp_path, contract):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    src, exe = str(tmp_path / "log_uniform.cpp"), str(tmp_path / "log_uniform")
    with open(src, "w") as f:
        f.write(SOURCE)
    flags = ["-mfma"] if "fma" in open("/proc/cpuinfo").read() else []
    subprocess.run([cxx, "-std=c++17", "-O2", "-w", "-ffp-contract=" + contract, "-D__HIP_PLATFORM_AMD__", "-I",
                    os.path.join(rocm, "include"), "-I", os.path.join(ROOT, "spirit_amd", "csrc"), src, "-o", exe] + flags,
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split()[0]) > 5 * 10 ** 6
