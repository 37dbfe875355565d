// The FP32 matrix-core detect of few samples: a tile's dictionary entries shared out over waves.
//
// A call of M samples is M / 32 waves of the whole-dictionary kernel, each a serial chain over all
// entries; up to 16384 samples that leaves half of the SIMDs without work and the others with one
// wave. Here a workgroup takes 64 samples and every wave a quarter (64 antennas: half) of the entries.
// What it costs is that a workgroup stages the dictionary for 64 samples instead of 128.
#include "apsm_detect_mfma.h"

namespace apsm {

template <int NMAX, int UMAX>
__global__ void __launch_bounds__( partsThreads( NMAX ), 2 ) apsm_detect_parts( const DetDesc x )
{
    detectTileMfma<NMAX, UMAX, PREC_F32, partsThreads( NMAX ) / 64, partsEntries( NMAX ), partsOf( NMAX )>(
        x.rx, x.M, x.Z, x.Zn, x.C, x.ldC, x.theta, x.G, x.U, x.wL, x.wG, x.g2, x.est, x.N, blockIdx.x );
}

template <int NMAX, int UMAX>
__global__ void __launch_bounds__( UMAX <= 4 ? kMfmaThreads : partsThreads( NMAX ), 2 )
    batch_detect_parts( const DetDesc* __restrict__ d, const WorkItem* __restrict__ items, int nItems )
{
    for ( int w = blockIdx.x; w < nItems; w += gridDim.x )
    {
        const WorkItem it = items[ w ];
        const DetDesc& x = d[ it.desc ];
        if constexpr ( UMAX <= 4 ) // batchWholeParts
            detectTileMfma<NMAX, UMAX, PREC_F32, kMfmaThreads / 64, 0, 1, partsOf( NMAX )>( x.rx, x.M, x.Z, x.Zn, x.C, x.ldC, x.theta, x.G, x.U,
                                                                                          x.wL, x.wG, x.g2, x.est, x.N, it.tile );
        else
            detectTileMfma<NMAX, UMAX, PREC_F32, partsThreads( NMAX ) / 64, partsEntries( NMAX ), partsOf( NMAX )>(
                x.rx, x.M, x.Z, x.Zn, x.C, x.ldC, x.theta, x.G, x.U, x.wL, x.wG, x.g2, x.est, x.N, it.tile );
    }
}

namespace {

// One launcher for both: a batch (items) or one handle's call.
struct PartsArgs
{
    hipStream_t s;
    const DetDesc* d;
    const WorkItem* items;
    int nItems, grid;
    DetDesc one;
};

template <int NMAX, int UMAX>
hipError_t launchNU( const PartsArgs& a )
{
    if ( a.items )
        hipLaunchKernelGGL( ( batch_detect_parts<NMAX, UMAX> ), dim3( a.grid ), dim3( batchPartsThreads( NMAX, UMAX ) ), 0, a.s, a.d, a.items,
                            a.nItems );
    else
        hipLaunchKernelGGL( ( apsm_detect_parts<NMAX, UMAX> ), dim3( (unsigned)( ( a.one.M + kPartsSamples - 1 ) / kPartsSamples ) ),
                            dim3( partsThreads( NMAX ) ), 0, a.s, a.one );
    return hipGetLastError();
}

template <int NMAX>
hipError_t launchN( int umax, const PartsArgs& a )
{
    switch ( umax )
    {
    case 1: return launchNU<NMAX, 1>( a );
    case 2: return launchNU<NMAX, 2>( a );
    case 4: return launchNU<NMAX, 4>( a );
    case 8: return launchNU<NMAX, 8>( a );
    case 12: return launchNU<NMAX, 12>( a );
    case 16: return launchNU<NMAX, 16>( a );
    default: return hipErrorInvalidValue;
    }
}

hipError_t launchAny( int nmax, int umax, const PartsArgs& a )
{
    switch ( nmax )
    {
    case 4: return launchN<4>( umax, a );
    case 8: return launchN<8>( umax, a );
    case 16: return launchN<16>( umax, a );
    case 32: return launchN<32>( umax, a );
    case 64: return launchN<64>( umax, a );
    default: return hipErrorInvalidValue;
    }
}

} // namespace

hipError_t launchDetectParts( int nmax, int umax, hipStream_t s, const DetDesc& x ) { return launchAny( nmax, umax, { s, nullptr, nullptr, 0, 0, x } ); }

hipError_t launchBatchDetectParts( int nmax, int umax, hipStream_t s, const DetDesc* d, const WorkItem* items, int nItems, int grid )
{
    return launchAny( nmax, umax, { s, d, items, nItems, grid, {} } );
}

} // namespace apsm
