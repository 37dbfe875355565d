// Shapes of the window sequencer (apsm_train_win.h) and the layout of what its block precompute
// writes for it. No kernels here: the Gram's translation unit includes it too.
#pragma once

#include "apsm_common.h"

namespace apsm {

constexpr int kWinTpCount = 6;
constexpr int kWinTps[ kWinTpCount ] = { 5, 10, 16, 20, 28, 40 }; // t-slots per lane: windowSize <= 4 TP

// t-slots per lane for a window of Wc complex samples (-1: none fits).
__host__ __device__ inline int winTp( int Wc )
{
    for ( int k = 0; k < kWinTpCount; k++ )
        if ( Wc <= 4 * kWinTps[ k ] )
            return kWinTps[ k ];
    return -1;
}

// Image of one sample's Gram column in slot order: 4 parts (16-lane rows) of three planes (A, C, B)
// of TPQ floats; parts padded to 16 bytes.
__host__ __device__ constexpr int winTpq( int tp ) { return ( tp + 1 ) & ~1; }
__host__ __device__ constexpr int winPart( int tp ) { return ( 3 * winTpq( tp ) + 3 ) & ~3; }
__host__ __device__ constexpr int winImg( int tp ) { return 4 * winPart( tp ); }
__host__ __device__ constexpr int winProductWaves( int tp ) { return ( 4 * tp + 15 ) / 16; }
// Helper waves: the packages with the window rows' share, and the left rows' share, 256 active samples
// per wave while the workgroup then has at most 8 waves (12 waves at TP = 40: 168 registers per
// wave, 120 of them the Gram).
__host__ __device__ constexpr int winLeftWaves( int tp ) { return tp <= 20 ? kActMax / 256 : 1; }
__host__ __device__ constexpr int winHelperWaves( int tp ) { return 1 + winLeftWaves( tp ); }
__host__ __device__ constexpr int winThreads( int tp ) { return 64 * ( winProductWaves( tp ) + winHelperWaves( tp ) ); }
// Package buffers: a package is issued BUFS - 2 steps before its first use, which has to cover the
// memory latency (about 1.2 us, four steps of the small windows).
constexpr int kWinBufs = 8;
// Left rows' kappa: register sets in flight of the helper that reads them (one per step).
__host__ __device__ constexpr int winRing( int tp ) { return tp <= 20 ? 4 : 2; }

// Block Gram buffer: Wc images of the window's samples at the block start (both orders of every
// pair), then one package row per entering sample e: its image over the window one step before it
// enters, 4 floats (kappa with itself: A, C, B, 0), and the kappa with the active samples that have
// left the window by then, three planes (A, kappa(a_e,b_j), kappa(b_e,a_j)) of ceil4(older) floats.
__host__ __device__ inline int winOlder( int e, int newRel0, int Wc )
{
    const int m = newRel0 + e - Wc;
    return m > 0 ? m : 0;
}
// sum of ceil4(o) over o < m
__host__ __device__ inline int winOlderSum( int m )
{
    if ( m < 2 )
        return 0;
    const int full = ( m - 1 ) >> 2, rem = ( m - 1 ) & 3;
    return 8 * full * ( full + 1 ) + 4 * rem * ( full + 1 );
}
__host__ __device__ inline int winRow( int e, int newRel0, int Wc, int tp )
{
    return Wc * winImg( tp ) + e * ( winImg( tp ) + 4 ) + 3 * winOlderSum( winOlder( e, newRel0, Wc ) );
}
// Floats of a block of `steps` steps (largest: a full window before the block), plus the last
// package copy's overrun (copies are whole 256-float chunks).
inline int64_t winGactFloats( int Wc, int steps )
{
    return (int64_t)winRow( steps, Wc - 1, Wc, winTp( Wc ) ) + 256;
}
// Row stride of the eviction shares [U][steps][stride], in slot order.
__host__ __device__ inline int winEvStride( int w2 ) { return ( w2 + 3 ) & ~3; }

// Package buffer in LDS: the image with the self entries, then the eviction shares, both in whole
// 256-float copies (the left rows' planes are not copied: their helper reads them from memory).
__host__ __device__ constexpr int winPkGram( int tp ) { return ( winImg( tp ) + 4 + 255 ) & ~255; }
__host__ __device__ constexpr int winPkEv( int tp ) { return ( 8 * tp + 255 ) & ~255; }
__host__ __device__ constexpr int winPkCap( int tp ) { return winPkGram( tp ) + winPkEv( tp ); }
// Floats of the eviction shares of U users in a block of `steps` steps, plus what the last row's copy
// reads beyond it: a row is shorter than the copy (228 floats against two pieces at windowSize 113).
inline int64_t winEvFloats( int64_t U, int64_t steps, int w2 )
{
    return U * steps * winEvStride( w2 ) + winPkEv( winTp( w2 / 2 ) );
}
// Beta pairs by t-slot, each 16-lane row's run padded to 16 bytes and so that the four rows' reads
// fall into different LDS banks; one more pair takes the writes of lanes without a t-slot.
__host__ __device__ constexpr int winBetaRun( int tp ) { return ( ( tp + 1 ) & ~1 ) + ( ( ( tp + 1 ) & ~1 ) % 16 == 0 ? 2 : 0 ); }
__host__ __device__ constexpr int winBetaFloats( int tp ) { return 8 * winBetaRun( tp ) + 4; }
inline size_t winLdsBytes( int tp )
{
    return sizeof( float ) * ( (size_t)kWinBufs * winPkCap( tp ) + 2 * winBetaFloats( tp ) + 2 * 32 * winProductWaves( tp ) + 2 * kActMax + 6 * ( kActMax + 2 ) + 4 * ( 1 + winLeftWaves( tp ) ) );
}

} // namespace apsm
