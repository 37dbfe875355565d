// Gram among the active samples of a train block on the matrix cores (FP32 inputs and
// accumulation), one block of the lower triangle per wave, four per workgroup.
//
// For two entering samples per step (gramBlockMfma): 32 x 32 blocks (rows i of block bi as the B
// operand, held in registers; rows j of block bj <= bi as the A operand, loaded from the stream buffer) of
// the two cross terms p = a_i.a_j and s = a_i.b_j with v_mfma_f32_32x32x2f32, written row by row. For the
// window sequencer (gramWinMfma): 16 x 16 blocks with v_mfma_f32_16x16x4f32, written in its layout.
#pragma once

#include "apsm_detect_mfma.h"
#include "apsm_win_layout.h"

namespace apsm {

typedef float f32x4 __attribute__( ( ext_vector_type( 4 ) ) );

template <int NMAX>
__device__ __forceinline__ void gramBlockMfma( const float* __restrict__ Z, const float* __restrict__ Zn, float* __restrict__ Gact,
                                               const GramArgs& a, const int64_t blk )
{
    constexpr int K = 2 * NMAX;
    const int N = a.N, L = a.L;
    const int lane = threadIdx.x & 63;
    const int col = lane & 31, h = lane >> 5;
    // block (bi, bj), bj <= bi, from the linear lower-triangle index
    int64_t bi = (int64_t)( ( sqrt( 8.0 * (double)blk + 1.0 ) - 1.0 ) * 0.5 );
    while ( ( bi + 1 ) * ( bi + 2 ) / 2 <= blk )
        bi++;
    while ( bi * ( bi + 1 ) / 2 > blk )
        bi--;
    const int64_t bj = blk - bi * ( bi + 1 ) / 2;
    const int64_t i = bi * 32 + col; // this lane's row (B operand column)
    const int64_t jr = bj * 32 + col; // the row this lane supplies as A operand
    const bool vi = i < a.nA, vj = jr < a.nA;
    const float* xi = Z + ( a.c0 + i ) * L;
    const float* zj = Z + ( a.c0 + jr ) * L;

    // operands first (all loads in flight at once), then the MFMA chain
    float xv[ K / 2 ], zr[ K / 2 ], zim[ K / 2 ];
#pragma unroll
    for ( int t = 0; t < K / 2; t++ )
    {
        const int k = 2 * t + h;
        const int ant = k < NMAX ? k : k - NMAX;
        xv[ t ] = ( ant < N && vi ) ? xi[ k < NMAX ? ant : N + ant ] : 0.f;
        zr[ t ] = ( ant < N && vj ) ? zj[ ant ] : 0.f;
        zim[ t ] = ( ant < N && vj ) ? zj[ N + ant ] : 0.f;
    }
    mf32x16 accP = {}, accS = {};
#pragma unroll
    for ( int t = 0; t < K / 2; t++ )
    {
        const bool re = 2 * t + h < NMAX;
        const float zp = re ? zr[ t ] : zim[ t ]; // Zp row = [Re z | Im z]
        const float zs = re ? zim[ t ] : -zr[ t ]; // Zs row = [Im z | -Re z]
        accP = __builtin_amdgcn_mfma_f32_32x32x2f32( zp, xv[ t ], accP, 0, 0, 0 );
        accS = __builtin_amdgcn_mfma_f32_32x32x2f32( zs, xv[ t ], accS, 0, 0, 0 );
    }
    if ( !vi )
        return;
    const float g2 = a.g2, k2 = 2.f * g2;
    const float qi = -g2 * Zn[ a.c0 + i ];
    const int64_t rowBase = gramRow( i );
#pragma unroll
    for ( int v = 0; v < 16; v++ )
    {
        const int64_t j = bj * 32 + 8 * ( v / 4 ) + 4 * h + ( v % 4 );
        if ( j > i || j >= a.nA )
            continue;
        const float q = qi - g2 * Zn[ a.c0 + j ];
        const float p = accP[ v ], s = accS[ v ];
        const float E0 = __builtin_amdgcn_exp2f( fminf( fmaf( k2, p, q ), 0.f ) );
        const float E1 = __builtin_amdgcn_exp2f( fminf( fmaf( k2, s, q ), 0.f ) );
        const float E2 = __builtin_amdgcn_exp2f( fminf( fmaf( -k2, s, q ), 0.f ) );
        float* o = Gact + rowBase + 3 * j;
        o[ 0 ] = a.wL * p + a.wG * E0;
        o[ 1 ] = a.wL * s + a.wG * E1;
        o[ 2 ] = -a.wL * s + a.wG * E2;
    }
}

// The same values in the window sequencer's layout (apsm_train_win.h). Here the rows i are the A
// operand and the rows j the B operand, so that the lanes of a store run along j, which is along
// an image's slots: the stores are contiguous but for the slots' wrap.
//
// Few waves, each a chain of loads, products, exponentials and stores, bound this: blocks of 16 x 16
// (v_mfma_f32_16x16x4_f32, four pairs per lane) give four times the waves of 32 x 32 ones, and all loads
// are issued before the first use.
template <int NMAX>
__device__ __forceinline__ void gramWinMfma( const float* __restrict__ Z, const float* __restrict__ Zn, float* __restrict__ Gact,
                                             const GramArgs& a, const int64_t blk )
{
    constexpr int T = NMAX / 4; // steps of four antennas
    const int N = a.N, L = a.L, Wc = a.Wc, tp = a.tp, nA = (int)a.nA, newRel0 = a.newRel0;
    const int lane = threadIdx.x & 63;
    const int r = lane & 15, g = lane >> 4;
    int bi = (int)( ( sqrtf( 8.f * (float)blk + 1.f ) - 1.f ) * 0.5f );
    while ( ( bi + 1 ) * ( bi + 2 ) / 2 <= blk )
        bi++;
    while ( bi * ( bi + 1 ) / 2 > blk )
        bi--;
    const int bj = (int)blk - bi * ( bi + 1 ) / 2;
    const int ir = bi * 16 + r; // the row this lane supplies as A operand
    const int j = bj * 16 + r; // this lane's B operand column
    const bool vi = ir < nA, vj = j < nA;
    const float* xi = Z + ( a.c0 + ir ) * L;
    const float* zj = Z + ( a.c0 + j ) * L;
    float xr[ T ], xm[ T ], zr[ T ], zm[ T ], ni[ 4 ];
#pragma unroll
    for ( int t = 0; t < T; t++ )
    {
        const int n = 4 * t + g;
        xr[ t ] = n < N && vi ? xi[ n ] : 0.f;
        xm[ t ] = n < N && vi ? xi[ N + n ] : 0.f;
        zr[ t ] = n < N && vj ? zj[ n ] : 0.f;
        zm[ t ] = n < N && vj ? zj[ N + n ] : 0.f;
    }
    const int i0 = bi * 16 + 4 * g; // this lane's pairs: (i0 + v, j)
#pragma unroll
    for ( int v = 0; v < 4; v++ )
        ni[ v ] = Zn[ a.c0 + ( i0 + v < nA ? i0 + v : nA - 1 ) ];
    const float nj = Zn[ a.c0 + ( vj ? j : nA - 1 ) ];
    f32x4 accP = { 0.f, 0.f, 0.f, 0.f }, accS = { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
    for ( int t = 0; t < T; t++ )
    {
        accP = __builtin_amdgcn_mfma_f32_16x16x4f32( xr[ t ], zr[ t ], accP, 0, 0, 0 );
        accS = __builtin_amdgcn_mfma_f32_16x16x4f32( xr[ t ], zm[ t ], accS, 0, 0, 0 );
        accP = __builtin_amdgcn_mfma_f32_16x16x4f32( xm[ t ], zm[ t ], accP, 0, 0, 0 );
        accS = __builtin_amdgcn_mfma_f32_16x16x4f32( -xm[ t ], zr[ t ], accS, 0, 0, 0 );
    }
    const int img = winImg( tp ), part = winPart( tp ), tpq = winTpq( tp );
    const float g2 = a.g2, k2 = 2.f * g2;
    const float qj = -g2 * nj;
    const int sj = ( a.cMod + j ) % Wc;
    const int oj = ( sj / tp ) * part + sj % tp; // this column's place in an image
#pragma unroll
    for ( int v = 0; v < 4; v++ )
    {
        const int i = i0 + v;
        const float q = qj - g2 * ni[ v ];
        const float p = accP[ v ], s = accS[ v ];
        const float E0 = __builtin_amdgcn_exp2f( fminf( fmaf( k2, p, q ), 0.f ) );
        const float E1 = __builtin_amdgcn_exp2f( fminf( fmaf( k2, s, q ), 0.f ) );
        const float E2 = __builtin_amdgcn_exp2f( fminf( fmaf( -k2, s, q ), 0.f ) );
        const float kA = a.wL * p + a.wG * E0; // kappa(a_i,a_j) = kappa(b_i,b_j)
        const float kB = a.wL * s + a.wG * E1; // kappa(a_i,b_j)
        const float kC = -a.wL * s + a.wG * E2; // kappa(b_i,a_j)
        if ( j > i || i >= nA )
            continue;
        if ( i < newRel0 )
        {
            // both in the window at the block start: the image of j (t = i) and the image of i (t = j)
            const int si = ( a.cMod + i ) % Wc;
            float* o = Gact + sj * img + ( si / tp ) * part + si % tp;
            o[ 0 ] = kA;
            o[ tpq ] = kC;
            o[ 2 * tpq ] = kB;
            o = Gact + si * img + oj;
            o[ 0 ] = kA;
            o[ tpq ] = kB;
            o[ 2 * tpq ] = kC;
        }
        else
        {
            const int e = i - newRel0;
            float* o = Gact + winRow( e, newRel0, Wc, tp );
            if ( i == j )
            {
                o[ img ] = kA;
                o[ img + 1 ] = kC;
                o[ img + 2 ] = kB;
            }
            else if ( i - j <= Wc )
            {
                o[ oj ] = kA;
                o[ oj + tpq ] = kB;
                o[ oj + 2 * tpq ] = kC;
            }
            else
            {
                const int o4 = ( winOlder( e, newRel0, Wc ) + 3 ) & ~3;
                o += img + 4 + j;
                o[ 0 ] = kA;
                o[ o4 ] = kB;
                o[ 2 * o4 ] = kC;
            }
        }
    }
    if ( bi != bj )
        return;
    // what a package row holds besides pairs: zeros in the image for slots without an active sample
    // and past the window, and in the padding of the older planes (all are multiplied by zero
    // coefficients, so they must be finite); 16 lanes per row
    for ( int i = bi * 16 + g; i < bi * 16 + 16 && i < nA; i += 4 )
    {
        if ( i < newRel0 )
            continue;
        const int e = i - newRel0;
        float* o = Gact + winRow( e, newRel0, Wc, tp );
        for ( int n = r; n < Wc - i; n += 16 )
        {
            const int sl = ( a.cMod + Wc - 1 - n ) % Wc; // relative sample -1 - n
            float* z = o + ( sl / tp ) * part + sl % tp;
            z[ 0 ] = z[ tpq ] = z[ 2 * tpq ] = 0.f;
        }
        for ( int sl = Wc + r; sl < 4 * tp; sl += 16 )
        {
            float* z = o + ( sl / tp ) * part + sl % tp;
            z[ 0 ] = z[ tpq ] = z[ 2 * tpq ] = 0.f;
        }
        const int older = winOlder( e, newRel0, Wc ), o4 = ( older + 3 ) & ~3;
        if ( r < 3 )
            for ( int n = older; n < o4; n++ )
                o[ img + 4 + r * o4 + n ] = 0.f;
    }
}

} // namespace apsm
