// Frozen-dictionary share of the entering pilots of one train block, with the cross terms on
// the matrix cores (FP32 inputs as three bf16 parts each, FP32 accumulation: the detect's core).
//
// For the entering complex samples i < nNewC of a block (rows newC0 + i of the stream buffer)
// and every user u: g_u(i) = sum over frozen dictionary entries j in [j0(i), j1) of
// (c_a E0 + c_b E1, c_a E2 + c_b E0), where j1 is the block's frozen boundary and j0(i) the
// dictionary's lower end when sample i enters (the FIFO may already have dropped entries).
// The frozen range is cut into chunks of kEntryChunk entries counted from its top (chunk 0 holds
// the most recently frozen entries); one workgroup takes one chunk
// for 128 entering samples, as the matrix-core detect (4 waves x 32 samples) does, masks the entries below j0(i), and writes its partial sums. A second kernel adds the
// chunks in order and the linear share: P_u(i) = wL thF_u.x_i + wG g_u(i).
#pragma once

#include "apsm_detect_mfma.h"
#include "apsm_gram_mfma.h"

namespace apsm {

template <int NMAX, int UMAX>
__device__ __forceinline__ void entryChunkMfma( const float* __restrict__ Z, const float* __restrict__ Zn, const float* __restrict__ C,
                                                float* __restrict__ part, const EntryArgs& a, const int64_t jBeg, const int nChunks,
                                                const int work )
{
    // work item = (tile of kMfmaSamples entering samples, chunk of the frozen range)
    const int chunk = work % nChunks, mBase = ( work / nChunks ) * kMfmaSamples;
    const int N = a.N, L = a.L;
    const int h = ( threadIdx.x >> 5 ) & 1;
    const int m = mBase + ( threadIdx.x >> 6 ) * 32 + ( threadIdx.x & 31 ); // entering sample of this lane
    const bool valid = m < a.nNewC;

    // dictionary lower end when sample m enters (entries below it are masked)
    const int64_t tc = a.newC0 + m;
    const int64_t rt = a.rowBase + 2 * tc;
    const int64_t se = rt < a.sFirst ? a.sFirst : a.sFirst + a.q * ( ( rt - a.sFirst ) / a.q + 1 );
    const int64_t lo = se > a.H ? se - a.H : 0;
    const int64_t jlo = ( lo - a.rowBase ) / 2;
    const int64_t j1 = ( a.a0 - a.rowBase ) / 2;

    // chunks from the top of the frozen range: chunk 0 holds the most recently frozen entries
    const int64_t c1 = j1 - (int64_t)chunk * kEntryChunk;
    const int64_t c0 = ( c1 - kEntryChunk ) > jBeg ? c1 - kEntryChunk : jBeg;
    const float* x = Z + tc * L;
    gaussianMfma<NMAX, UMAX, PREC_F32, kMfmaThreads / 64, 0, true, 1, 1>(
        Z + c0 * L, Zn + c0, C + 2 * c0, a.ldYC, c1 - c0, a.U, a.g2, N,
        [ & ]( int n ) { return valid && n < N ? make_float2( x[ n ], x[ N + n ] ) : make_float2( 0.f, 0.f ); },
        [ & ]( int64_t j0 ) { // entries of the tile from j0 that the FIFO dropped before this lane's sample entered
            const int64_t d = jlo - c0 - j0;
            return d < 0 ? 0 : d > kEntryChunk ? (int)kEntryChunk : (int)d;
        },
        [ & ]( float( &fa )[ UMAX ], float( &fb )[ UMAX ] ) {
            if ( !valid || h != 0 )
                return;
#pragma unroll
            for ( int u = 0; u < UMAX; u++ )
                if ( u < a.U )
                    reinterpret_cast<float2*>( part )[ ( (int64_t)u * nChunks + chunk ) * a.nNewC + m ] = make_float2( fa[ u ], fb[ u ] );
        } );
}

// P_u(i) = wL thF_u.x_i + wG (sum of the chunk partials): 64 (u, i) per workgroup, 16 slices of the
// antennas and of the chunks, whose sums are added in order. (One thread per (u, i) waited for
// the chunks one after another.)
constexpr int kCombineSlices = 16, kCombineThreads = 64 * kCombineSlices;
__device__ __forceinline__ void entryCombineBody( const float* __restrict__ Z, const float* __restrict__ thF, const float* __restrict__ part,
                                                  float* __restrict__ P, const EntryArgs& a, const int nChunks, const int wg )
{
    __shared__ float4 sum[ kCombineSlices ][ 64 ];
    const int col = threadIdx.x & 63, slice = threadIdx.x >> 6;
    const int idx = wg * 64 + col;
    const int N = a.N;
    float la = 0.f, lb = 0.f, ga = 0.f, gb = 0.f;
    if ( idx < a.U * a.nNewC )
    {
        const int u = idx / a.nNewC, i = idx % a.nNewC;
        const float* x = Z + ( a.newC0 + i ) * a.L;
        const float* th = thF + (int64_t)u * a.L;
#pragma unroll 4
        for ( int n = slice; n < N; n += kCombineSlices )
        {
            const float xr = x[ n ], xi = x[ N + n ];
            la += fmaf( th[ n ], xr, th[ N + n ] * xi );
            lb += fmaf( th[ n ], xi, -th[ N + n ] * xr );
        }
        const float2* pp = reinterpret_cast<const float2*>( part ) + (int64_t)u * nChunks * a.nNewC + i;
#pragma unroll 8
        for ( int c = slice; c < nChunks; c += kCombineSlices )
        {
            const float2 v = pp[ (int64_t)c * a.nNewC ];
            ga += v.x;
            gb += v.y;
        }
    }
    sum[ slice ][ col ] = make_float4( la, lb, ga, gb );
    __syncthreads();
    if ( slice != 0 || idx >= a.U * a.nNewC )
        return;
#pragma unroll
    for ( int k = 1; k < kCombineSlices; k++ )
    {
        const float4 v = sum[ k ][ col ];
        la += v.x;
        lb += v.y;
        ga += v.z;
        gb += v.w;
    }
    reinterpret_cast<float2*>( P )[ idx ] = make_float2( a.wL * la + a.wG * ga, a.wL * lb + a.wG * gb );
}

template <int NMAX, int UMAX>
__global__ void __launch_bounds__( kMfmaThreads, 2 ) apsm_entry_mfma( const float* __restrict__ Z, const float* __restrict__ Zn,
                                                                  const float* __restrict__ C, float* __restrict__ part, const EntryArgs a,
                                                                  int64_t jBeg, int nChunks, int chunk0 )
{
    entryChunkMfma<NMAX, UMAX>( Z, Zn, C, part, a, jBeg, nChunks, chunk0 + blockIdx.x );
}

__global__ void __launch_bounds__( kCombineThreads ) apsm_entry_combine( const float* __restrict__ Z, const float* __restrict__ thF, const float* __restrict__ part,
                                    float* __restrict__ P, const EntryArgs a, int nChunks )
{
    entryCombineBody( Z, thF, part, P, a, nChunks, blockIdx.x );
}

__global__ void __launch_bounds__( kCombineThreads ) batch_entry_combine( const EntryMfmaDesc* __restrict__ d )
{
    const EntryMfmaDesc& e = d[ blockIdx.y ];
    if ( (int)blockIdx.x * 64 < e.a.U * e.a.nNewC )
        entryCombineBody( e.Z, e.thF, e.part, e.P, e.a, e.nChunks, blockIdx.x );
}

// What a further block of a train call costs besides its steps (precompute, combine, launches; 8
// antennas, at windowSize 20 / 40 / 80 / 160): 17 / 24 / 25 / 36 us with FP32 products of 32 x 32 blocks, one load
// at a time and a serial combine, 11 / 12 / 13 / 21 us now. Latency bounds it: a few hundred waves, each
// one chain.
//
// One block's precompute, workgroup b: entry work item (the first entryWg workgroups), Gram
// blocks (the next gramWg) or eviction shares (the last evWg); batched: gridX = the largest sum.
template <int NMAX, int UMAX>
__device__ __forceinline__ void blockPreBody( const PreDesc& d, int b )
{
    if ( b < d.entryWg )
    {
        entryChunkMfma<NMAX, UMAX>( d.e.Z, d.e.Zn, d.e.C, d.e.part, d.e.a, d.e.jBeg, d.e.nChunks, b );
        return;
    }
    b -= d.entryWg;
    if ( b < d.gramWg )
    {
        const int64_t blk = (int64_t)b * ( kMfmaThreads / 64 ) + ( threadIdx.x >> 6 );
        if ( blk < gramBlocks( d.g.a ) )
        {
            if ( d.g.a.Wc )
                gramWinMfma<NMAX>( d.g.Z, d.g.Zn, d.g.Gact, d.g.a, blk );
            else
                gramBlockMfma<NMAX>( d.g.Z, d.g.Zn, d.g.Gact, d.g.a, blk );
        }
        return;
    }
    b -= d.gramWg;
    if ( b < d.evWg )
        evictCorrBody( d.v.Z, d.v.Zn, d.v.C, d.v.EvF, d.v.a, (int64_t)b * kMfmaThreads + threadIdx.x );
}

template <int NMAX, int UMAX>
__global__ void __launch_bounds__( kMfmaThreads, 2 ) apsm_block_pre( const PreDesc d )
{
    blockPreBody<NMAX, UMAX>( d, blockIdx.x );
}

template <int NMAX, int UMAX>
__global__ void __launch_bounds__( kMfmaThreads, 2 ) batch_block_pre( const PreDesc* __restrict__ d )
{
    const PreDesc& x = d[ blockIdx.y ];
    if ( (int)blockIdx.x >= x.entryWg + x.gramWg + x.evWg )
        return;
    blockPreBody<NMAX, UMAX>( x, blockIdx.x );
}

template <int NMAX, int UMAX>
hipError_t launchPreNU( bool batch, hipStream_t s, const PreDesc* d, int n, int gridX )
{
    if ( batch )
        hipLaunchKernelGGL( ( batch_block_pre<NMAX, UMAX> ), dim3( gridX, n ), dim3( kMfmaThreads ), 0, s, d );
    else
        hipLaunchKernelGGL( ( apsm_block_pre<NMAX, UMAX> ), dim3( gridX ), dim3( kMfmaThreads ), 0, s, *d );
    return hipGetLastError();
}

template <int NMAX>
hipError_t launchPreN( int umax, bool batch, hipStream_t s, const PreDesc* d, int n, int gridX )
{
    switch ( umax )
    {
    case 1: return launchPreNU<NMAX, 1>( batch, s, d, n, gridX );
    case 2: return launchPreNU<NMAX, 2>( batch, s, d, n, gridX );
    case 4: return launchPreNU<NMAX, 4>( batch, s, d, n, gridX );
    case 8: return launchPreNU<NMAX, 8>( batch, s, d, n, gridX );
    case 12: return launchPreNU<NMAX, 12>( batch, s, d, n, gridX );
    case 16: return launchPreNU<NMAX, 16>( batch, s, d, n, gridX );
    default: return hipErrorInvalidValue;
    }
}

inline hipError_t launchPreAnyN( int nmax, int umax, bool batch, hipStream_t s, const PreDesc* d, int n, int gridX )
{
    switch ( nmax )
    {
    case 4: return launchPreN<4>( umax, batch, s, d, n, gridX );
    case 8: return launchPreN<8>( umax, batch, s, d, n, gridX );
    case 16: return launchPreN<16>( umax, batch, s, d, n, gridX );
    case 32: return launchPreN<32>( umax, batch, s, d, n, gridX );
    case 64: return launchPreN<64>( umax, batch, s, d, n, gridX );
    default: return hipErrorInvalidValue;
    }
}

// Entry work items [chunk0, chunk0 + count) of one block of a single handle.
template <int NMAX, int UMAX>
hipError_t launchEntryNU( hipStream_t s, const float* Z, const float* Zn, const float* C, float* part, const EntryArgs& a, int64_t jBeg,
                          int nChunks, int chunk0, int count )
{
    hipLaunchKernelGGL( ( apsm_entry_mfma<NMAX, UMAX> ), dim3( count ), dim3( kMfmaThreads ), 0, s, Z, Zn, C, part, a, jBeg, nChunks, chunk0 );
    return hipGetLastError();
}

template <int NMAX>
hipError_t launchEntryN( int umax, hipStream_t s, const float* Z, const float* Zn, const float* C, float* part, const EntryArgs& a,
                         int64_t jBeg, int nChunks, int chunk0, int count )
{
    switch ( umax )
    {
    case 1: return launchEntryNU<NMAX, 1>( s, Z, Zn, C, part, a, jBeg, nChunks, chunk0, count );
    case 2: return launchEntryNU<NMAX, 2>( s, Z, Zn, C, part, a, jBeg, nChunks, chunk0, count );
    case 4: return launchEntryNU<NMAX, 4>( s, Z, Zn, C, part, a, jBeg, nChunks, chunk0, count );
    case 8: return launchEntryNU<NMAX, 8>( s, Z, Zn, C, part, a, jBeg, nChunks, chunk0, count );
    case 12: return launchEntryNU<NMAX, 12>( s, Z, Zn, C, part, a, jBeg, nChunks, chunk0, count );
    case 16: return launchEntryNU<NMAX, 16>( s, Z, Zn, C, part, a, jBeg, nChunks, chunk0, count );
    default: return hipErrorInvalidValue;
    }
}

inline hipError_t launchEntryAnyN( int nmax, int umax, hipStream_t s, const float* Z, const float* Zn, const float* C, float* part,
                                   const EntryArgs& a, int64_t jBeg, int nChunks, int chunk0, int count )
{
    switch ( nmax )
    {
    case 4: return launchEntryN<4>( umax, s, Z, Zn, C, part, a, jBeg, nChunks, chunk0, count );
    case 8: return launchEntryN<8>( umax, s, Z, Zn, C, part, a, jBeg, nChunks, chunk0, count );
    case 16: return launchEntryN<16>( umax, s, Z, Zn, C, part, a, jBeg, nChunks, chunk0, count );
    case 32: return launchEntryN<32>( umax, s, Z, Zn, C, part, a, jBeg, nChunks, chunk0, count );
    case 64: return launchEntryN<64>( umax, s, Z, Zn, C, part, a, jBeg, nChunks, chunk0, count );
    default: return hipErrorInvalidValue;
    }
}

} // namespace apsm
