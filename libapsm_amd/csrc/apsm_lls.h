// Least squares over the real embedding (cpp/lib/noma/lls_detector.cu:136-218): min_w |A w - y| with
// rows a = [Re x | Im x], b = [Im x | -Re x] of every pilot, by the normal equations in FP64.
//
// Between antennas u and v the normal matrix holds two different sums only,
//   P = sum re_u re_v + im_u im_v  (Re-Re and Im-Im),  Q = sum re_u im_v - im_u re_v  (Re-Im; antisymmetric),
// and with y in the place of x_u they are the right-hand side.
#pragma once

#include "apsm_common.h"

#include <type_traits>

namespace apsm {

typedef double f64x4 __attribute__( ( ext_vector_type( 4 ) ) );

// ---- normal matrix: P and Q of 16 x 16 antennas over a share of the pilots ----------------------
constexpr int kLlsPairThreads = 256;  // four waves, each a quarter of the share
constexpr int kLlsPairEntries = 512;  // P and Q of one pair of antenna blocks
constexpr int64_t kLlsMinShare = 128; // pilots per workgroup: 8 steps of 4 pilots per wave
constexpr int64_t kLlsShares = 128;   // at most: partial sums of 64 antennas stay below 8 MB

__host__ __device__ constexpr int llsBlocks( int N ) { return ( N + 15 ) / 16; }
// pairs of antenna blocks (lower triangle), then y with every block
__host__ __device__ constexpr int llsTasks( int N ) { return llsBlocks( N ) * ( llsBlocks( N ) + 3 ) / 2; }
inline int64_t llsShare( int64_t T )
{
    const int64_t s = ( T + kLlsShares - 1 ) / kLlsShares;
    return s <= kLlsMinShare ? kLlsMinShare : ( s + 31 ) / 32 * 32; // whole steps of eight pilots per wave
}

// Block pair of task q: rows from block ib (llsBlocks(N): y), columns from block jb.
__device__ __forceinline__ void llsPairOf( int q, int nb, int& ib, int& jb )
{
    const int pairs = nb * ( nb + 1 ) / 2;
    if ( q >= pairs )
    {
        ib = nb;
        jb = q - pairs;
        return;
    }
    ib = 0;
    while ( ( ib + 1 ) * ( ib + 2 ) / 2 <= q )
        ib++;
    jb = q - ib * ( ib + 1 ) / 2;
}

// Grid (shares, tasks). FP32 pilots, exact FP64 products, FP64 sums on the FP64 matrix cores
// (v_mfma_f64_16x16x4, 64 cycles, bounds the kernel: 4 per pair and 4 pilots). Lane l feeds row or
// column l % 16 of pilots 2 * (l / 16) + {0, 1} of every eight.
__global__ void __launch_bounds__( kLlsPairThreads ) lls_normal_pairs( const float* __restrict__ rx, const float* __restrict__ tx,
                                                                     int N, int64_t T, int64_t share, double* __restrict__ part )
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int nb = llsBlocks( N );
    int ib, jb;
    llsPairOf( blockIdx.y, nb, ib, jb );
    const float2* x = reinterpret_cast<const float2*>( rx );
    const int ri = 16 * ib + r, rj = 16 * jb + r;
    const bool hasI = ib < nb ? ri < N : r == 0, hasJ = rj < N;
    const float2* pi = ib < nb ? x + (int64_t)( hasI ? ri : 0 ) * T : reinterpret_cast<const float2*>( tx );
    const float2* pj = x + (int64_t)( hasJ ? rj : 0 ) * T;
    const int64_t k0 = (int64_t)blockIdx.x * share + wave * ( share / 4 );
    const int64_t k1 = k0 + share / 4 < T ? k0 + share / 4 : T;
    f64x4 P = { 0., 0., 0., 0. }, Q = { 0., 0., 0., 0. };
#pragma unroll 4
    for ( int64_t k = k0; k < k1; k += 8 )
    {
        const int64_t t = k + 2 * g;
        float2 a[ 2 ], b[ 2 ];
#pragma unroll
        for ( int e = 0; e < 2; e++ )
        {
            a[ e ] = hasI && t + e < k1 ? pi[ t + e ] : make_float2( 0.f, 0.f );
            b[ e ] = hasJ && t + e < k1 ? pj[ t + e ] : make_float2( 0.f, 0.f );
        }
#pragma unroll
        for ( int e = 0; e < 2; e++ )
        {
            P = __builtin_amdgcn_mfma_f64_16x16x4f64( (double)a[ e ].x, (double)b[ e ].x, P, 0, 0, 0 );
            Q = __builtin_amdgcn_mfma_f64_16x16x4f64( (double)a[ e ].x, (double)b[ e ].y, Q, 0, 0, 0 );
            P = __builtin_amdgcn_mfma_f64_16x16x4f64( (double)a[ e ].y, (double)b[ e ].y, P, 0, 0, 0 );
            Q = __builtin_amdgcn_mfma_f64_16x16x4f64( -(double)a[ e ].y, (double)b[ e ].x, Q, 0, 0, 0 );
        }
    }
    __shared__ double sum[ 3 ][ kLlsPairEntries ];
    // result layout: column l % 16, row 4 v + l / 16
    if ( wave > 0 )
#pragma unroll
        for ( int v = 0; v < 4; v++ )
        {
            sum[ wave - 1 ][ 64 * v + lane ] = P[ v ];
            sum[ wave - 1 ][ 256 + 64 * v + lane ] = Q[ v ];
        }
    __syncthreads();
    if ( wave == 0 )
    {
        double* out = part + ( (int64_t)blockIdx.x * gridDim.y + blockIdx.y ) * kLlsPairEntries;
#pragma unroll
        for ( int v = 0; v < 4; v++ )
        {
            const int e = 64 * v + lane; // = 16 * row + column
            out[ e ] = P[ v ] + sum[ 0 ][ e ] + sum[ 1 ][ e ] + sum[ 2 ][ e ];
            out[ 256 + e ] = Q[ v ] + sum[ 0 ][ 256 + e ] + sum[ 1 ][ 256 + e ] + sum[ 2 ][ 256 + e ];
        }
    }
}

// ---- sums of partials: 64 entries per workgroup, 16 slices of the partials -----------------------
constexpr int kLlsSumThreads = 1024;
template <class T>
__device__ __forceinline__ double llsSumPartials( const T* __restrict__ part, int nPart, int64_t stride, bool ok )
{
    __shared__ double s[ 16 ][ 64 ];
    const int e = threadIdx.x & 63, slice = threadIdx.x >> 6;
    double v = 0.0;
    if ( ok )
#pragma unroll 8
        for ( int b = slice; b < nPart; b += 16 )
            v += (double)part[ b * stride ];
    s[ slice ][ e ] = v;
    __syncthreads();
    v = 0.0;
    if ( slice == 0 )
#pragma unroll
        for ( int k = 0; k < 16; k++ )
            v += s[ k ][ e ];
    return v; // slice 0
}

// Grid (tasks, 8): the pair sums as the lower triangle and the right-hand side of G, [L][L+1].
__global__ void __launch_bounds__( kLlsSumThreads ) lls_reduce_pairs( const double* __restrict__ part, int nPart, int N,
                                                                    double* __restrict__ G )
{
    const int e = 64 * blockIdx.y + ( threadIdx.x & 63 );
    const double v = llsSumPartials( part + (int64_t)blockIdx.x * kLlsPairEntries + e, nPart, (int64_t)gridDim.x * kLlsPairEntries, true );
    if ( threadIdx.x >= 64 )
        return;
    const int nb = llsBlocks( N ), L = 2 * N, ld = L + 1;
    int ib, jb;
    llsPairOf( blockIdx.x, nb, ib, jb );
    const bool isQ = e >= 256;
    const int i = ( e & 255 ) >> 4, b = 16 * jb + ( e & 15 ), a = 16 * ib + i;
    if ( b >= N )
        return;
    if ( ib == nb )
    {
        if ( i == 0 )
            G[ ( isQ ? N + b : b ) * ld + L ] = v;
    }
    else if ( a < N && !isQ )
    {
        if ( a >= b )
        {
            G[ a * ld + b ] = v;
            G[ ( N + a ) * ld + N + b ] = v;
        }
    }
    else if ( a < N )
    {
        G[ ( N + a ) * ld + b ] = -v;
        if ( ib > jb )
            G[ ( N + b ) * ld + a ] = v;
    }
}

// G[e] = sum of FP32 partials in FP64; grid ceil(E / 64).
__global__ void __launch_bounds__( kLlsSumThreads ) lls_reduce_partials( const float* __restrict__ part, int nPart, int E,
                                                                       double* __restrict__ G )
{
    const int e = blockIdx.x * 64 + ( threadIdx.x & 63 );
    const double v = llsSumPartials( part + e, nPart, E, e < E );
    if ( threadIdx.x < 64 && e < E )
        G[ e ] = v;
}

// ---- solve ----------------------------------------------------------------------------------
// G = R D R^T (unit lower triangular R) and R D R^T w = r in FP64, L <= 16 NB unknowns; G is
// [L][L+1] with the right-hand side in column L, its lower triangle is read. Writes w (FP32) and the
// status: 0 ok, -1 a column is empty, a pivot negative, or more than two columns (one antenna) depend on
// the others.
//
// A pivot counts as kSolveFloor of its diagonal entry at least. What is left of a column that depends on
// the others is rounding: its inputs', 2^-48 of the entry and less, or the sums'. Divided by that,
// the weights are of 1e6, which FP32 estimates do not survive, or the pivot's sign refuses the system by
// chance (x_1 = a x_0 + x_2, 4 antennas, 200 pilots, noise 0.07: residual up to 0.84, 0.074 with the
// floor; two equal antennas: 3 of 100 solved, all with the floor).
//
// The serial chain of L columns bounds it (LDS round trip, barrier, reciprocal), so a column is one
// barrier: thread (ty, tx) keeps the entries (ty + 16 p, tx + 16 q) in registers, the owners of column j put
// it, not yet divided by its pivot, into LDS as R's column times the pivot, and every thread
// reads what its own entries need. No square roots; the right-hand side is one more row. The back
// substitution is one wave's, a column at a time.
constexpr int kSolveThreads = 256;
constexpr double kSolveFloor = 0x1p-32; // (weights then stay below 2^16 |y| / |x_j|)
__host__ __device__ constexpr int llsSolveBlocks( int L ) { return L <= 16 ? 1 : L <= 32 ? 2 : L <= 64 ? 4 : 8; }
constexpr size_t llsSolveLds( int L ) { return (size_t)L * ( 16 * llsSolveBlocks( L ) + 1 ) * sizeof( double ); }

__device__ __forceinline__ double readLaneF64( double v, int lane )
{
    const uint64_t u = __builtin_bit_cast( uint64_t, v );
    const uint32_t lo = __builtin_amdgcn_readlane( (uint32_t)u, lane ), hi = __builtin_amdgcn_readlane( (uint32_t)( u >> 32 ), lane );
    return __builtin_bit_cast( double, (uint64_t)hi << 32 | lo );
}

template <int NB>
__global__ void __launch_bounds__( kSolveThreads ) lls_solve( const double* __restrict__ Gin, int L, float* __restrict__ w,
                                                            int* __restrict__ status )
{
    constexpr int ld = 16 * NB + 1; // odd; the last entry of a column is the right-hand side's
    extern __shared__ double col[]; // [L][ld]
    __shared__ double sInv[ 16 * NB ], sFloor[ 16 * NB ];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    double a[ NB ][ NB ], z[ NB ];
    auto factor = [ & ]( auto floorC ) {
#pragma unroll
        for ( int p = 0; p < NB; p++ )
#pragma unroll
            for ( int q = 0; q <= p; q++ )
            {
                const int i = ty + 16 * p, k = tx + 16 * q;
                a[ p ][ q ] = i < L && k <= i ? Gin[ i * ( L + 1 ) + k ] : 0.0;
                if ( p == q && tx == ty )
                    sFloor[ i ] = a[ p ][ q ] > 0.0 ? kSolveFloor * a[ p ][ q ] : -1.0; // negative: an empty column
            }
#pragma unroll
        for ( int q = 0; q < NB; q++ )
            z[ q ] = tx + 16 * q < L ? Gin[ ( tx + 16 * q ) * ( L + 1 ) + L ] : 0.0;
#pragma unroll
        for ( int jb = 0; jb < NB; jb++ )
#pragma unroll 1
            for ( int jj = 0; jj < 16; jj++ )
            {
                const int j = 16 * jb + jj;
                if ( j >= L )
                    break;
                double* cj = col + j * ld;
                if ( tx == jj )
                {
#pragma unroll
                    for ( int p = jb; p < NB; p++ )
                        cj[ ty + 16 * p ] = a[ p ][ jb ];
                    if ( ty == 0 )
                        cj[ ld - 1 ] = z[ jb ];
                }
                __syncthreads();
                double d = cj[ j ], zj = cj[ ld - 1 ], ci[ NB ], ck[ NB ];
#pragma unroll
                for ( int p = jb; p < NB; p++ )
                {
                    ci[ p ] = cj[ ty + 16 * p ];
                    ck[ p ] = cj[ tx + 16 * p ];
                }
                if constexpr ( floorC )
                    d = fmax( d, fabs( sFloor[ j ] ) );
                double inv = __builtin_amdgcn_rcp( d ); // and two Newton steps
                inv = fma( fma( -d, inv, 1.0 ), inv, inv );
                inv = fma( fma( -d, inv, 1.0 ), inv, inv );
                if ( threadIdx.x == 0 )
                    sInv[ j ] = inv;
                // (rows and columns up to j of block jb are finished: what these get is not used)
#pragma unroll
                for ( int q = jb; q < NB; q++ )
                {
                    const double f = -ck[ q ] * inv;
                    z[ q ] = fma( f, zj, z[ q ] );
#pragma unroll
                    for ( int p = q; p < NB; p++ )
                        a[ p ][ q ] = fma( f, ci[ p ], a[ p ][ q ] );
                }
            }
        __syncthreads();
    };
    // The pivots are looked at afterwards, off the chain; a system with one below its floor is factored
    // once more with the floors.
    auto below = [ & ]( int k ) { return k < L && !( col[ k * ld + k ] >= sFloor[ k ] && sFloor[ k ] > 0.0 ); };
    factor( std::false_type {} );
    if ( __syncthreads_or( below( threadIdx.x ) ) )
        factor( std::true_type {} );
    if ( threadIdx.x < 64 )
    {
        // w_j = (z_j - sum_{i > j} col_j[i] w_i) / d_j: lane k keeps unknowns k and k + 64
        constexpr int H = NB > 4 ? 2 : 1;
        const int lane = threadIdx.x;
        double acc[ H ], x[ H ];
        bool bad = false;
        int dependent = 0;
#pragma unroll
        for ( int h = 0; h < H; h++ )
        {
            const int k = lane + 64 * h < L ? lane + 64 * h : 0;
            acc[ h ] = col[ k * ld + ld - 1 ];
            x[ h ] = 0.0;
            const double d = col[ k * ld + k ], least = sFloor[ k ];
            bad |= least < 0.0 || !( d >= -least );
            dependent += __popcll( __ballot( lane + 64 * h < L && d < least ) );
        }
        bad = __ballot( bad ) != 0 || dependent > 2;
#pragma unroll
        for ( int hj = H - 1; hj >= 0; hj-- )
        {
            const int top = L - 64 * hj < 64 ? L - 64 * hj : 64;
#pragma unroll 8
            for ( int jl = top - 1; jl >= 0; jl-- )
            {
                const int j = 64 * hj + jl;
                const double wj = readLaneF64( acc[ hj ], jl ) * sInv[ j ];
                x[ hj ] = lane == jl ? wj : x[ hj ];
#pragma unroll
                for ( int h = 0; h <= hj; h++ )
                {
                    const int k = lane + 64 * h < L ? lane + 64 * h : 0; // (lanes from j on are finished)
                    acc[ h ] = fma( -col[ k * ld + j ], wj, acc[ h ] );
                }
            }
        }
#pragma unroll
        for ( int h = 0; h < H; h++ )
            if ( lane + 64 * h < L )
                w[ lane + 64 * h ] = (float)x[ h ];
        if ( lane == 0 )
            *status = bad ? -1 : 0;
    }
}

// est[m] = (a_m . w, b_m . w)  (lls_detector.cu:207-218, a GEMV over the embedding). Bounded by reading rx.
__global__ void lls_apply( const float* __restrict__ rx, int N, int64_t M, const float* __restrict__ w, float* __restrict__ est )
{
    const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if ( m >= M )
        return;
    float ea = 0.f, eb = 0.f;
    int n = 0;
    for ( ; n + 8 <= N; n += 8 )
    {
        float2 v[ 8 ]; // in flight together
#pragma unroll
        for ( int i = 0; i < 8; i++ )
            v[ i ] = reinterpret_cast<const float2*>( rx )[ (int64_t)( n + i ) * M + m ];
#pragma unroll
        for ( int i = 0; i < 8; i++ )
        {
            ea += v[ i ].x * w[ n + i ] + v[ i ].y * w[ N + n + i ];
            eb += v[ i ].y * w[ n + i ] - v[ i ].x * w[ N + n + i ];
        }
    }
    for ( ; n < N; n++ )
    {
        const float2 v = reinterpret_cast<const float2*>( rx )[ (int64_t)n * M + m ];
        ea += v.x * w[ n ] + v.y * w[ N + n ];
        eb += v.y * w[ n ] - v.x * w[ N + n ];
    }
    reinterpret_cast<float2*>( est )[ m ] = make_float2( ea, eb );
}

} // namespace apsm
