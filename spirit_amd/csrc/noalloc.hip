// Gradient and energy of caller-owned device spins without any device allocation.
//
// Spirit_HIP_Gradient_and_Energy builds a runner with its own device buffers (spins,
// gradient, pair tables, per-block partial sums) on every call.  Callers that cannot
// allocate device memory (code under graph capture, tight serving loops, harnesses that
// forbid hipMalloc) call Spirit_HIP_Gradient_and_Energy_NoAlloc instead: inputs and outputs
// are the caller's device arrays, and everything else the kernels need lives in `scratch`,
// a file-scope device array of fixed size that each GPU holds until the process ends.
//
// A call is one kernel for lattices of up to NA_FOLD_BLOCKS blocks of a nearest-neighbour model, two for
// larger ones: it reads and writes the caller's arrays as they are, its Hamiltonian is a kernel
// argument, and only tables that do not fit one are copied.
//
// Scratch layout (byte offsets): the counter of the blocks that have stored their energy (zero between
// calls), the pair and quadruplet tables, the per-block energy partials, the per-site K_i, and the
// gradient where the caller's arrays overlap.  Calls on one GPU share the array;
// the entry point holds a per-device lock until its stream has finished, so calls through it
// never overlap on one GPU, but any other user of the array would race with them.
#include "api_common.hpp"
#include "gpu_engine.hpp"
#include "llg_device.hpp"

#include <mutex>

namespace spirit_hip
{

namespace
{

constexpr long long NA_MAX_SPINS  = SPIRIT_HIP_NOALLOC_MAX_SPINS;
constexpr int NA_MAX_BLOCKS       = (int)( ( NA_MAX_SPINS + LLG_THREADS - 1 ) / LLG_THREADS );
constexpr int NA_MAX_PAIR_ENTRIES = 2 * MAX_PAIRS; // exchange + DMI
constexpr int NA_MAX_QUADS        = 512;
constexpr int NA_FOLD_BLOCKS      = 128; // blocks whose energies the gradient kernel adds itself

constexpr size_t align256( size_t x )
{
    return ( x + 255 ) / 256 * 256;
}
constexpr size_t OFF_COUNT  = 0;
constexpr size_t OFF_PAIRS  = align256( OFF_COUNT + sizeof( int ) );
constexpr size_t OFF_QUADS  = align256( OFF_PAIRS + sizeof( PairDev ) * NA_MAX_PAIR_ENTRIES );
constexpr size_t OFF_PART_E = align256( OFF_QUADS + sizeof( QuadDev ) * NA_MAX_QUADS );
constexpr size_t OFF_SITE_K = align256( OFF_PART_E + sizeof( double ) * NA_MAX_BLOCKS );
constexpr size_t OFF_G      = align256( OFF_SITE_K + sizeof( double ) * NA_MAX_SPINS );
constexpr size_t SCRATCH_BYTES = align256( OFF_G + sizeof( double ) * 3 * NA_MAX_SPINS );

} // namespace

// The scratch array.  In host code this name is only a stand-in for the symbol: host code
// uses the per-device address hipGetSymbolAddress returns (scratch_address below).
static __device__ __align__( 256 ) unsigned char scratch[SCRATCH_BYTES];

namespace
{

constexpr int NA_MAX_DEVICES = 64;

struct DeviceScratch
{
    std::mutex lock;     // held for a whole call: calls through the entry point never overlap
    char * ptr = nullptr; // address of this device's copy of `scratch`
};
DeviceScratch g_dev[NA_MAX_DEVICES];
std::mutex g_setup_lock;

// The address of the current device's copy of `scratch`, looked up once per device with that
// device current.
DeviceScratch & scratch_address( int & device )
{
    if( hipGetDevice( &device ) != hipSuccess )
        throw api_error( 1, "Spirit_HIP_Gradient_and_Energy_NoAlloc: no current HIP device" );
    if( device < 0 || device >= NA_MAX_DEVICES )
        throw api_error( 1, "Spirit_HIP_Gradient_and_Energy_NoAlloc: device index out of range" );
    DeviceScratch & d = g_dev[device];
    std::lock_guard<std::mutex> lk( g_setup_lock );
    if( !d.ptr )
    {
        void * p       = nullptr;
        hipError_t err = hipGetSymbolAddress( &p, HIP_SYMBOL( scratch ) );
        if( err != hipSuccess || !p )
            throw api_error( 1, std::string( "Spirit_HIP_Gradient_and_Energy_NoAlloc: hipGetSymbolAddress failed: " )
                                    + hipGetErrorString( err ) );
        d.ptr = static_cast<char *>( p );
    }
    return d;
}

// E = sum of the n block partials in block order, the order Spirit_HIP_Gradient_and_Energy adds them on
// the host, so both entry points return the same bits: the block brings them to LDS, thread 0 adds.
__device__ __forceinline__ void sum_partials( const double * part, int n, double * out )
{
    constexpr int CHUNK = 4 * LLG_THREADS;
    __shared__ double lds[CHUNK];
    double E = 0;
    for( int k0 = 0; k0 < n; k0 += CHUNK )
    {
        const int m = n - k0 < CHUNK ? n - k0 : CHUNK;
        for( int k = threadIdx.x; k < m; k += LLG_THREADS )
            lds[k] = __hip_atomic_load( part + k0 + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
        __syncthreads();
        if( threadIdx.x == 0 )
        {
#pragma unroll 8
            for( int k = 0; k < m; ++k )
                E += lds[k];
        }
        __syncthreads();
    }
    if( threadIdx.x == 0 )
        *out = E;
}

__global__ void __launch_bounds__( LLG_THREADS ) k_na_sum( const double * part, int n, double * out )
{
    sum_partials( part, n, out );
}

__global__ void __launch_bounds__( LLG_THREADS ) k_na_copy( const double * src, double * dst, long long n )
{
    const long long i = blockIdx.x * (long long)LLG_THREADS + threadIdx.x;
    if( i < n )
        dst[i] = src[i];
}

// Gradient of the spins x (an array of spins, like the gradient) and every block's energy; with out, the
// last block to arrive adds the energies (fold_finalize of the stage kernels has the protocol; with one
// counter 128 blocks take 1 us to arrive, 256 as long as a launch costs).  A call was bound by its launches and copies, not by this kernel: five
// kernels and two copies took 37.6 us for 64 x 64 spins, this one 22.8, of which the kernel is 10.
template<bool FEW>
__global__ void __launch_bounds__( LLG_THREADS )
    k_na_gradient( HamDev H, const double * __restrict__ x, double * __restrict__ grad, double * part, int * count,
                   double * out )
{
    const int blk = xcd_contiguous_block();
    const int i   = blk * LLG_THREADS + threadIdx.x;
    double e_i    = 0;
    if( i < H.nos )
    {
        double g[3];
        local_gradient<FEW, true>( H, x, H.nos, i, nullptr, g, e_i );
#pragma unroll
        for( int q = 0; q < 3; ++q )
            grad[3LL * i + q] = g[q];
    }
    __shared__ double sE[LLG_THREADS / 64];
    __shared__ int last;
    double t = 0;
    wave_reduce( e_i, t );
    if( threadIdx.x % 64 == 0 )
        sE[threadIdx.x / 64] = e_i;
    __syncthreads();
    if( threadIdx.x == 0 )
    {
        for( int k = 1; k < LLG_THREADS / 64; ++k )
            e_i += sE[k];
        __hip_atomic_store( part + blk, e_i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
        last = 0;
        if( out )
        {
            __builtin_amdgcn_fence( __ATOMIC_RELEASE, "workgroup" );
            __builtin_amdgcn_s_waitcnt( 0 ); // the store is performed
            last = __hip_atomic_fetch_add( count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT ) == (int)gridDim.x - 1;
        }
    }
    __syncthreads();
    if( !last )
        return;
    if( threadIdx.x == 0 )
        __hip_atomic_store( count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
    sum_partials( part, gridDim.x, out );
}

// whether n doubles at p and m doubles at q have memory in common
bool overlap( const double * p, long long n, const double * q, long long m )
{
    return (uintptr_t)p < (uintptr_t)( q + m ) && (uintptr_t)q < (uintptr_t)( p + n );
}

void check( hipError_t e, const char * what )
{
    if( e != hipSuccess )
        throw api_error( 1, std::string( "Spirit_HIP_Gradient_and_Energy_NoAlloc: " ) + what + ": "
                                + hipGetErrorString( e ) );
}

} // namespace

} // namespace spirit_hip

using namespace spirit_hip;

extern "C" int Spirit_HIP_Gradient_and_Energy_NoAlloc( State * state, const double * spins, double * gradient,
                                                      double * energy, void * stream, int idx_image,
                                                      int idx_chain ) noexcept
try
{
    std::shared_ptr<Image> image;
    std::shared_ptr<Chain> chain;
    from_indices( state, idx_image, idx_chain, image, chain );
    if( !spins || !gradient || !energy )
        throw api_error( 2, "Spirit_HIP_Gradient_and_Energy_NoAlloc: spins, gradient and energy must be device arrays" );
    std::lock_guard<std::recursive_mutex> ilk( image->mtx );
    const Geometry & g    = *image->geometry;
    const Hamiltonian & h = *image->hamiltonian;
    const int nos         = g.nos;
    if( nos < 1 || nos > NA_MAX_SPINS )
        throw api_error( 2, "Spirit_HIP_Gradient_and_Energy_NoAlloc: " + std::to_string( nos )
                                + " spins, the limit is " + std::to_string( NA_MAX_SPINS ) );
    if( h.ddi_method != DDI_NONE )
        throw api_error( 2, "Spirit_HIP_Gradient_and_Energy_NoAlloc: dipolar interactions need the DDI plan's "
                            "buffers; use Spirit_HIP_Gradient_and_Energy" );
    if( h.exch_pairs.size() + h.dmi_pairs.size() > (size_t)NA_MAX_PAIR_ENTRIES )
        throw api_error( 2, "Spirit_HIP_Gradient_and_Energy_NoAlloc: more than " + std::to_string( NA_MAX_PAIR_ENTRIES )
                                + " exchange and DMI pairs" );
    if( h.quads.size() > (size_t)NA_MAX_QUADS )
        throw api_error( 2, "Spirit_HIP_Gradient_and_Energy_NoAlloc: more than " + std::to_string( NA_MAX_QUADS )
                                + " quadruplets" );

    int device         = 0;
    DeviceScratch & ds = scratch_address( device );
    std::lock_guard<std::mutex> dlk( ds.lock );
    char * base           = ds.ptr;
    const hipStream_t st  = static_cast<hipStream_t>( stream );
    const int n_blocks    = ( nos + LLG_THREADS - 1 ) / LLG_THREADS;
    int * d_count         = reinterpret_cast<int *>( base + OFF_COUNT );
    PairDev * d_pairs     = reinterpret_cast<PairDev *>( base + OFF_PAIRS );
    QuadDev * d_quads     = reinterpret_cast<QuadDev *>( base + OFF_QUADS );
    double * d_part_E     = reinterpret_cast<double *>( base + OFF_PART_E );
    double * d_site_K     = reinterpret_cast<double *>( base + OFF_SITE_K );
    double * d_g          = reinterpret_cast<double *>( base + OFF_G );

    // the Hamiltonian and its tables, built on the host stack; tables that are no part of it are copied
    // into the scratch
    PairDev pairs[NA_MAX_PAIR_ENTRIES];
    QuadDev quads[NA_MAX_QUADS];
    HamDev H{};
    const int n_pairs = fill_ham_dev( g, h, H, pairs, NA_MAX_PAIR_ENTRIES );
    H.exch        = d_pairs;
    H.dmi         = d_pairs + H.n_exch;
    const int n_quads = (int)h.quads.size();
    for( int k = 0; k < n_quads; ++k )
    {
        const Quadruplet & q = h.quads[k];
        if( q.i < 0 || q.i >= g.nb || q.j < 0 || q.j >= g.nb || q.k < 0 || q.k >= g.nb || q.l < 0 || q.l >= g.nb )
            throw api_error( 2, "Spirit_HIP_Gradient_and_Energy_NoAlloc: quadruplet with a basis index outside the cell" );
        QuadDev d{};
        d.i = q.i, d.j = q.j, d.k = q.k, d.l = q.l;
        for( int c = 0; c < 3; ++c )
        {
            d.dj[c] = q.dj[c];
            d.dk[c] = q.dk[c];
            d.dl[c] = q.dl[c];
        }
        d.Q      = h.quad_Q[k];
        quads[k] = d;
    }
    if( n_quads > 0 )
    {
        H.n_quad       = n_quads;
        H.quad_in_step = h.quadruplets_in_gradient_and_energy() ? 1 : 0;
        H.quad         = d_quads;
    }
    if( H.has_site_K )
        H.site_K = d_site_K;

    const bool few = few_pairs( H );
    if( n_pairs > 0 && !few )
        check( hipMemcpyAsync( d_pairs, pairs, sizeof( PairDev ) * n_pairs, hipMemcpyHostToDevice, st ),
               "copy of the pair table" );
    if( n_quads > 0 )
        check( hipMemcpyAsync( d_quads, quads, sizeof( QuadDev ) * n_quads, hipMemcpyHostToDevice, st ),
               "copy of the quadruplets" );
    if( H.has_site_K )
        check( hipMemcpyAsync( d_site_K, h.site_K.data(), sizeof( double ) * nos, hipMemcpyHostToDevice, st ),
               "copy of the per-site anisotropy" );
    // arrays that share memory: the gradient is formed beside them and copied, the energy stored last
    const bool apart = !overlap( spins, 3LL * nos, gradient, 3LL * nos ) && !overlap( spins, 3LL * nos, energy, 1 )
                       && !overlap( gradient, 3LL * nos, energy, 1 );
    const bool fold  = apart && n_blocks <= NA_FOLD_BLOCKS;
    hipLaunchKernelGGL( few ? k_na_gradient<true> : k_na_gradient<false>, dim3( n_blocks ), dim3( LLG_THREADS ), 0, st,
                        H, spins, apart ? gradient : d_g, d_part_E, d_count, fold ? energy : nullptr );
    if( !apart )
        hipLaunchKernelGGL( k_na_copy, dim3( ( 3 * nos + LLG_THREADS - 1 ) / LLG_THREADS ), dim3( LLG_THREADS ), 0, st,
                            d_g, gradient, 3LL * nos );
    if( !fold )
        hipLaunchKernelGGL( k_na_sum, dim3( 1 ), dim3( LLG_THREADS ), 0, st, d_part_E, n_blocks, energy );
    check( hipGetLastError(), "kernel launch" );
    // the host-side tables above are read by the copies: wait for the stream before they go
    check( hipStreamSynchronize( st ), "stream synchronisation" );
    return 0;
}
catch( ... )
{
    handle_exception( idx_image, idx_chain );
    return 1;
}
