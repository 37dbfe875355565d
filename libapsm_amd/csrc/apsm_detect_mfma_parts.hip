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

namespace {

template <int NMAX, int UMAX>
hipError_t launchNU( hipStream_t s, const DetDesc& x )
{
    hipLaunchKernelGGL( ( apsm_detect_parts<NMAX, UMAX> ), dim3( (unsigned)( ( x.M + kPartsSamples - 1 ) / kPartsSamples ) ),
                        dim3( partsThreads( NMAX ) ), 0, s, x );
    return hipGetLastError();
}

template <int NMAX>
hipError_t launchN( int umax, hipStream_t s, const DetDesc& x )
{
    switch ( umax )
    {
    case 1: return launchNU<NMAX, 1>( s, x );
    case 2: return launchNU<NMAX, 2>( s, x );
    case 4: return launchNU<NMAX, 4>( s, x );
    case 8: return launchNU<NMAX, 8>( s, x );
    case 12: return launchNU<NMAX, 12>( s, x );
    case 16: return launchNU<NMAX, 16>( s, x );
    default: return hipErrorInvalidValue;
    }
}

} // namespace

hipError_t launchDetectParts( int nmax, int umax, hipStream_t s, const DetDesc& x )
{
    switch ( nmax )
    {
    case 4: return launchN<4>( umax, s, x );
    case 8: return launchN<8>( umax, s, x );
    case 16: return launchN<16>( umax, s, x );
    case 32: return launchN<32>( umax, s, x );
    case 64: return launchN<64>( umax, s, x );
    default: return hipErrorInvalidValue;
    }
}

} // namespace apsm
