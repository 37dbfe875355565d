// Detect with the cross terms on the matrix cores.
//
// For data samples x (columns) and dictionary entries z (rows) the two real cross terms are
// the GEMMs  P^T = Zp X^T  and  S^T = Zp Xs^T  with K = 2*NMAX (zero padded):
//   Zp row = [Re z | Im z],  X row = [Re x | Im x],  Xs row = [-Im x | Re x],
// so p = a_x.a_z and s = a_x.b_z. One wave computes a 32 entries x 32 samples block of each
// with v_mfma_f32_32x32x16_{bf16,f16}, FP32 accumulation. In the result layout lane l holds
// sample l % 32 and the 16 entries 8*(v/4) + 4*(l/32) + v%4 (v = 0..15), so the rest of the pair
// work stays in the lane: squared distances from the FP32 norms |x|^2 + |z|^2 (the norm
// correction is FP32 for every precision), three exponentials, and the contraction with every
// user's coefficients. The two lane halves hold disjoint entries of the same sample and are added
// at the end.
//
// PREC_BF16 and PREC_F16 round the inputs to 16 bits. PREC_F32 cuts every input into three bf16
// parts, v = h + m + l (8 bits each: all 24 of an FP32 mantissa), and sums the six products above
// 2^-24, hl, mm, lh, hm, mh, hh, smallest first: exact products, FP32 accumulation, so the error is
// that of an FP32 dot product (the dropped ml, lm, ll are below 2^-25 of |x||z|). Six bf16 products
// of 16 components take 192 cycles against 512 for v_mfma_f32_32x32x2_f32, and unlike those (which
// share the vector ALU's multipliers) they run beside the vector ALU's exponentials.
//
// Workgroup: WAVES waves x 32 samples; the dictionary streams through LDS in tiles of ETILE entries.
// The vector ALU's share per block of 32 x 32 pairs is 16 x (3 exponentials of 8.2 cycles, which take
// the clamp at 1 for free, 4 + 4 U multiply-adds and adds of about 4 between them): 900 cycles for one
// user, against 12 matrix instructions of 32 cycles up to 8 antennas, 24 at 16, 48 at 32. The next
// block's products run between this one's exponentials, so what bounds a block is the power limit: with both units busy
// the clock falls from 2.1 GHz to 1.6 to 1.75. Detect calls before (FP32 products on
// v_mfma_f32_32x32x2_f32, one block's products and exponentials after each other) and now:
//   8 antennas, 685 centres, 3840 samples              60 -> 33 us
//   16 antennas, 10 users, 4096 centres, 500k samples  5.69 -> 3.38 ms
//   32 antennas, 3690 centres, 49999 samples           678 -> 279 us
//   64 antennas, 12 users, 16384 centres, 400k samples, bf16  16.1 -> 13.0 ms
// or per block of 32 x 32 and SIMD, in cycles as if at 2.4 GHz: 1460 (8 antennas), 2070 (16), 3340 (32), 6880 (64),
// measured with one sum per user; kept by parts (ORDER) within 4 % of that.
// Measured and not kept: two column blocks per wave sharing the coefficient reads (10 % faster at 4 users,
// slower elsewhere, 64 antennas spilled); 8 waves per workgroup (within 2 %); staging loads without
// the bounds branches (20 % slower); all products before all exponentials (as fast up to 16
// antennas, 64 antennas bf16 8540 against 5810).
#pragma once

#include "apsm_detect_launch.h"

#include <utility>

namespace apsm {


typedef float mf32x16 __attribute__( ( ext_vector_type( 16 ) ) );
typedef __bf16 mbf16x8 __attribute__( ( ext_vector_type( 8 ) ) );
typedef _Float16 mf16x8 __attribute__( ( ext_vector_type( 8 ) ) );

template <int PREC>
struct MfmaIn;
template <>
struct MfmaIn<PREC_BF16>
{
    typedef __bf16 T;
    typedef mbf16x8 V;
    static __device__ __forceinline__ mf32x16 mma( V a, V b, mf32x16 c ) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16( a, b, c, 0, 0, 0 ); }
};
template <>
struct MfmaIn<PREC_F16>
{
    typedef _Float16 T;
    typedef mf16x8 V;
    static __device__ __forceinline__ mf32x16 mma( V a, V b, mf32x16 c ) { return __builtin_amdgcn_mfma_f32_32x32x16_f16( a, b, c, 0, 0, 0 ); }
};

template <>
struct MfmaIn<PREC_F32> : MfmaIn<PREC_BF16> // three bf16 parts
{
};

typedef float mf32x2 __attribute__( ( ext_vector_type( 2 ) ) );

// Two values as packed 16-bit inputs of the matrix cores: NS = 1 rounds, NS = 3 gives h, m, l.
template <int PREC, int NS>
__device__ __forceinline__ void mfmaParts( float v0, float v1, uint32_t ( &out )[ NS ] )
{
    typedef typename MfmaIn<PREC>::T T2 __attribute__( ( ext_vector_type( 2 ) ) );
    mf32x2 v = { v0, v1 };
#pragma unroll
    for ( int i = 0; i < NS; i++ )
    {
        const T2 q = __builtin_convertvector( v, T2 );
        out[ i ] = __builtin_bit_cast( uint32_t, q );
        if ( i + 1 < NS )
            v -= __builtin_convertvector( q, mf32x2 );
    }
}

// f( 0 ) ... f( N - 1 ) with the index as a constant expression
template <class F, int... I>
__device__ __forceinline__ void unrollSeq( F& f, std::integer_sequence<int, I...> )
{
    ( f( std::integral_constant<int, I> {} ), ... );
}
template <int N, class F>
__device__ __forceinline__ void unrollFor( F f )
{
    unrollSeq( f, std::make_integer_sequence<int, N> {} );
}

// The Gaussian part of f for 32 samples per wave over the dictionary entries [0, G) of Z, Zn, C:
// load( n ) is antenna n of this lane's sample (zero for none), finish( fa, fb ) takes every user's sums
// (for the lanes of the first half; the two halves of a wave hold disjoint entries of the same samples
// and have been added). MASK: entries below first( j0 ), counted within the tile from j0, do not count.
// WAVES: waves per workgroup; ETILE: dictionary entries per LDS tile (0: mfmaTileOf). PARTS > 1: the
// entries of a tile (32 PARTS) are shared out over PARTS waves of the same samples, wave w taking block
// w % PARTS, and finish is called for the first of them with the parts added in order. ORDER > 1: a wave
// takes all entries and adds the blocks b % ORDER up by themselves, which gives the bits of PARTS = ORDER:
// for few users side by side, otherwise in the order 0, ORDER, 2 ORDER, ..., 1, ORDER + 1, ... of the blocks,
// one run after another (from 6 users on the finished runs' sums wait in LDS, for the registers' sake).
template <int NMAX, int UMAX, int PREC, int WAVES, int ETILE, bool MASK, int PARTS, int ORDER, class LOAD, class FIRST, class FINISH>
__device__ __forceinline__ void gaussianMfma( const float* __restrict__ Z, const float* __restrict__ Zn, const float* __restrict__ C,
                                              int64_t ldC, int64_t G, int U, float g2, int N, LOAD load, FIRST first, FINISH finish )
{
    constexpr int K = 2 * NMAX, K16 = K < 16 ? 16 : K, T = K16 / 16; // components, padded; steps of 16
    constexpr int NS = PREC == PREC_F32 ? 3 : 1;
    constexpr int kTile = ETILE ? ETILE : mfmaTileOf( NMAX, PREC );
    constexpr int kThreads = 64 * WAVES;
    constexpr int RowH = K16 + 8; // rows padded by 16 bytes against LDS bank conflicts of the 16-byte reads
    constexpr int kAllQuads = K16 / 4 * kTile, kQuads = ( kAllQuads + kThreads - 1 ) / kThreads; // groups of four components staged per thread
    constexpr int kCLoads = ( UMAX * kTile + kThreads - 1 ) / kThreads;
    static_assert( kTile <= kThreads && kTile % 32 == 0, "staging shape" );
    static_assert( PARTS == 1 || ( kTile == 32 * PARTS && WAVES % PARTS == 0 && !MASK ), "one block per wave and tile" );
    static_assert( ORDER == 1 || ( !MASK && PARTS == 1 ), "runs of blocks are one wave's" );
    typedef typename MfmaIn<PREC>::V V;
    typedef uint32_t u32x4 __attribute__( ( ext_vector_type( 4 ) ) );
    // two tile buffers: the next tile's loads are in flight (in registers) while the current tile
    // is used, so a tile costs one barrier
    __shared__ __attribute__( ( aligned( 16 ) ) ) uint16_t sZ[ 2 ][ NS ][ kTile * RowH ];
    __shared__ __attribute__( ( aligned( 16 ) ) ) float sZn[ 3 ][ kTile ];
    __shared__ __attribute__( ( aligned( 16 ) ) ) float2 sC[ 3 ][ kTile * UMAX ]; // [entry][user]
    // Few users: all ORDER sums in registers and the blocks in plain order, block b in sum b % ORDER; else one run after
    // another. By runs a tile's rows are not consecutive and every block may end one: up to 4 % (512 detectors
    // as a batch, one user each: detect 47.6 ms by runs, 42.4 side by side). At 32 antennas and two users the
    // sums spill, and from 6 users on they do not fit; at 64 antennas runs are as fast.
    constexpr bool KEEP = ORDER > 1 && NMAX <= 32 && ( UMAX == 1 || ( UMAX <= 4 && NMAX <= 16 ) ), RUNS = ORDER > 1 && !KEEP;
    constexpr int SUMS = KEEP ? ORDER : 1;
    constexpr bool SUMLDS = RUNS && UMAX > 4;
    __shared__ float sSum[ SUMLDS ? UMAX * 64 * WAVES : 1 ]; // [user][lane]: sums of the finished runs

    const int tid = threadIdx.x, lane = tid & 63;
    const int col = lane & 31, h = lane >> 5;
    const int L = 2 * N;

    // This lane's half of the sample as B operands: step t holds components 16t + 8h + i of X and Xs.
    // A component pair (re, im) of an antenna is one 8-byte load; with NMAX a multiple of 16 the Re
    // half of X is the second half of Xs, and only the negated Im half is kept besides X. At 64
    // antennas in three parts not even that fits the registers: the products with Im x go to an
    // accumulator of their own and are subtracted.
    constexpr bool HALVES = NMAX % 16 == 0, SUBTRACT = NMAX >= 64 && NS == 3;
    constexpr int TX = SUBTRACT ? 1 : HALVES ? T / 2 : T; // steps of Xs with registers of their own
    V xp[ T ][ NS ], xs[ TX ][ NS ];
    float xq; // -g2 |x|^2
    {
        float xn = 0.f;
        if constexpr ( HALVES )
        {
#pragma unroll
            for ( int t = 0; t < T / 2; t++ )
            {
                u32x4 re[ NS ], im[ NS ];
#pragma unroll
                for ( int i = 0; i < 8; i += 2 )
                {
                    float2 v[ 2 ];
#pragma unroll
                    for ( int e = 0; e < 2; e++ )
                    {
                        const int ant = 16 * t + 8 * h + i + e;
                        v[ e ] = load( ant );
                        xn += v[ e ].x * v[ e ].x + v[ e ].y * v[ e ].y;
                    }
                    uint32_t pr[ NS ], pi[ NS ];
                    mfmaParts<PREC, NS>( v[ 0 ].x, v[ 1 ].x, pr );
                    mfmaParts<PREC, NS>( v[ 0 ].y, v[ 1 ].y, pi );
#pragma unroll
                    for ( int q = 0; q < NS; q++ )
                    {
                        re[ q ][ i / 2 ] = pr[ q ];
                        im[ q ][ i / 2 ] = pi[ q ];
                    }
                }
#pragma unroll
                for ( int q = 0; q < NS; q++ )
                {
                    xp[ t ][ q ] = __builtin_bit_cast( V, re[ q ] );
                    xp[ t + T / 2 ][ q ] = __builtin_bit_cast( V, im[ q ] );
                    if constexpr ( !SUBTRACT )
                        xs[ t ][ q ] = __builtin_bit_cast( V, im[ q ] ^ 0x80008000u );
                }
            }
            xn += __shfl_xor( xn, 32 );
        }
        else
        {
            // NMAX 8: half h = 0 holds Re x, h = 1 Im x; NMAX 4: half 0 holds both, half 1 is padding
            u32x4 p4[ NS ], s4[ NS ];
#pragma unroll
            for ( int i = 0; i < 8; i += 2 )
            {
                float vp[ 2 ], vs[ 2 ];
#pragma unroll
                for ( int e = 0; e < 2; e++ )
                {
                    const int ant = ( i + e ) % NMAX;
                    const float2 v = load( ant );
                    if ( NMAX == 8 || i < 4 )
                        xn += v.x * v.x + v.y * v.y;
                    const bool lo = NMAX == 8 ? h == 0 : i < 4; // component of Re x
                    const float keep = NMAX == 8 || h == 0 ? 1.f : 0.f;
                    vp[ e ] = keep * ( lo ? v.x : v.y );
                    vs[ e ] = keep * ( lo ? -v.y : v.x );
                }
                uint32_t pp[ NS ], ps[ NS ];
                mfmaParts<PREC, NS>( vp[ 0 ], vp[ 1 ], pp );
                mfmaParts<PREC, NS>( vs[ 0 ], vs[ 1 ], ps );
#pragma unroll
                for ( int q = 0; q < NS; q++ )
                {
                    p4[ q ][ i / 2 ] = pp[ q ];
                    s4[ q ][ i / 2 ] = ps[ q ];
                }
            }
#pragma unroll
            for ( int q = 0; q < NS; q++ )
            {
                xp[ 0 ][ q ] = __builtin_bit_cast( V, p4[ q ] );
                xs[ 0 ][ q ] = __builtin_bit_cast( V, s4[ q ] );
            }
        }
        xq = -g2 * xn;
    }
    // exponent arguments with the scale folded in: -g2 * (|x|^2 + |z|^2 - 2p) = q + k2 * p; the
    // constants in vector registers (a scalar operand halves the multiply-add's rate)
    float k2 = 2.f * g2, k2n = -2.f * g2;
    asm( "" : "+v"( k2 ), "+v"( k2n ) );

    float fa[ SUMS ][ UMAX ], fb[ SUMS ][ UMAX ];
    auto addHalves = [ & ]() {
#pragma unroll
        for ( int o = 0; o < SUMS; o++ )
#pragma unroll
            for ( int u = 0; u < UMAX; u++ )
            {
                fa[ o ][ u ] += __shfl_xor( fa[ o ][ u ], 32 );
                fb[ o ][ u ] += __shfl_xor( fb[ o ][ u ], 32 );
            }
    };
    float sum[ SUMLDS ? 1 : UMAX ]; // sums of the finished runs, fa's in lane half 0 and fb's in 1
    float* const sums = sSum + ( SUMLDS ? tid : 0 );
#pragma unroll
    for ( int u = 0; u < UMAX; u++ )
    {
#pragma unroll
        for ( int o = 0; o < SUMS; o++ )
            fa[ o ][ u ] = fb[ o ][ u ] = 0.f;
        if ( SUMLDS )
            sums[ u * 64 * WAVES ] = 0.f;
        else
            sum[ u ] = 0.f;
    }

    const int nBlocks = (int)( ( G + 31 ) / 32 );

    // tile loads into registers (zeros past the dictionary end, past N and past K): components k to k + 3
    // of entry e, r * kThreads + tid = e * K16/4 + k/4. With N == NMAX rows have no gaps: one 16-byte load.
    // A tile holds the next blocks of the order taken.
    constexpr int kTileBlocks = kTile / 32;
    static_assert( kTileBlocks <= 2 || kTileBlocks == 4, "blockOf" );
    int bLoad = 0, runLoad = 0; // next block to load, its run
    const float* zLoad = Z; // and its first row
    auto nextBlock = [ & ]() { // of the runs
        const int b = bLoad;
        bLoad += ORDER;
        if ( bLoad >= nBlocks )
        {
            runLoad++;
            bLoad = runLoad < ORDER ? runLoad : nBlocks;
        }
        return b;
    };
    float4 zreg[ kQuads ];
    float zn;
    float2 creg[ kCLoads ];
    const bool whole = N == NMAX && K == K16 && ( reinterpret_cast<uintptr_t>( Z ) & 15 ) == 0;
    auto loadRows = [ & ]() { // a tile of consecutive rows
        const int64_t j0 = (int64_t)( RUNS ? nextBlock() : bLoad ) * 32;
        if ( !RUNS )
            bLoad += kTileBlocks;
        const int nt = ( G - j0 ) < kTile ? (int)( G - j0 ) : kTile;
        if ( whole )
        {
            const float4* Zt = reinterpret_cast<const float4*>( Z + j0 * L );
#pragma unroll
            for ( int r = 0; r < kQuads; r++ )
            {
                const int i = r * kThreads + tid;
                zreg[ r ] = i / ( K16 / 4 ) < nt ? Zt[ i ] : make_float4( 0.f, 0.f, 0.f, 0.f );
            }
        }
        else
        {
#pragma unroll
            for ( int r = 0; r < kQuads; r++ )
            {
                const int i = r * kThreads + tid;
                const int k = 4 * ( i % ( K16 / 4 ) ), e = i / ( K16 / 4 );
                const int n = k < NMAX ? k : k - NMAX;
                const float* z = Z + ( j0 + e ) * L + ( k < NMAX ? n : N + n );
                const int have = e < nt && k < K ? N - n : 0;
                zreg[ r ].x = have > 0 ? z[ 0 ] : 0.f;
                zreg[ r ].y = have > 1 ? z[ 1 ] : 0.f;
                zreg[ r ].z = have > 2 ? z[ 2 ] : 0.f;
                zreg[ r ].w = have > 3 ? z[ 3 ] : 0.f;
            }
        }
        zn = tid < nt ? -g2 * Zn[ j0 + tid ] : 0.f;
#pragma unroll
        for ( int r = 0; r < kCLoads; r++ )
        {
            const int i = r * kThreads + tid;
            const int u = i / kTile, e = i % kTile;
            creg[ r ] = ( i < UMAX * kTile && u < U && e < nt )
                ? make_float2( C[ u * ldC + 2 * ( j0 + e ) ], C[ u * ldC + 2 * ( j0 + e ) + 1 ] )
                : make_float2( 0.f, 0.f );
        }
    };
    auto loadBlocks = [ & ]() { // a tile of the next blocks of the runs
        int blk[ kTileBlocks ];
        const float* row[ kTileBlocks ]; // their first rows
        unrollFor<kTileBlocks>( [ & ]( auto iC ) {
            row[ iC ] = zLoad;
            const int run = runLoad;
            blk[ iC ] = nextBlock();
            zLoad = runLoad == run ? zLoad + ORDER * 32 * L : Z + (int64_t)bLoad * 32 * L;
        } );
        // element i (of values: selects of elements would keep the array in memory)
        auto pick = [ & ]( const auto& v, int i ) {
            const auto v0 = v[ 0 ], v1 = v[ kTileBlocks > 1 ? 1 : 0 ], v2 = v[ kTileBlocks > 2 ? 2 : 0 ], v3 = v[ kTileBlocks - 1 ];
            const auto lo = i < 1 ? v0 : v1, hi = i < 3 ? v2 : v3;
            return kTileBlocks < 4 || i < 2 ? lo : hi;
        };
        const int Gi = (int)G;
        constexpr int kBlockQuads = 8 * K16; // a wave's quads lie in one block
#pragma unroll
        for ( int r = 0; r < kQuads; r++ )
        {
            const int bi = __builtin_amdgcn_readfirstlane( ( r * kThreads + tid ) / kBlockQuads ), i = r * kThreads + tid - bi * kBlockQuads;
            const int e = i / ( K16 / 4 );
            const int nt = kAllQuads % kThreads != 0 && bi >= kTileBlocks ? 0 : Gi - 32 * pick( blk, bi ); // (32 and more: a whole block)
            const float* z0 = pick( row, bi );
            if ( whole )
                zreg[ r ] = e < nt ? reinterpret_cast<const float4*>( z0 )[ i ] : make_float4( 0.f, 0.f, 0.f, 0.f );
            else
            {
                const int k = 4 * ( i % ( K16 / 4 ) );
                const int n = k < NMAX ? k : k - NMAX;
                const float* z = z0 + e * L + ( k < NMAX ? n : N + n );
                const int have = e < nt && k < K ? N - n : 0;
                zreg[ r ].x = have > 0 ? z[ 0 ] : 0.f;
                zreg[ r ].y = have > 1 ? z[ 1 ] : 0.f;
                zreg[ r ].z = have > 2 ? z[ 2 ] : 0.f;
                zreg[ r ].w = have > 3 ? z[ 3 ] : 0.f;
            }
        }
        static_assert( kThreads % kTile == 0, "a thread stages one entry's norm and coefficients" );
        const int j = pick( blk, tid % kTile / 32 ) * 32 + tid % 32;
        const bool in = j < Gi;
        zn = tid < kTile && in ? -g2 * Zn[ j ] : 0.f;
#pragma unroll
        for ( int r = 0; r < kCLoads; r++ )
        {
            const int u = r * ( kThreads / kTile ) + tid / kTile;
            // (C and ldC are even numbers of floats from an allocation's start)
            creg[ r ] = u < UMAX && u < U && in ? reinterpret_cast<const float2*>( C + u * ldC )[ j ] : make_float2( 0.f, 0.f );
        }
    };
    auto loadTile = [ & ]() {
        if constexpr ( RUNS && ( kTileBlocks > 1 || UMAX > 8 || ( NMAX >= 64 && UMAX > 2 ) ) ) // (scalar addresses: fewer spills)
            loadBlocks();
        else
            loadRows();
    };
    auto storeTile = [ & ]( int tt ) {
        const int buf = tt & 1, slot = tt % 3;
#pragma unroll
        for ( int r = 0; r < kQuads; r++ )
        {
            const int i = r * kThreads + tid;
            const int k = 4 * ( i % ( K16 / 4 ) ), e = i / ( K16 / 4 );
            if ( kAllQuads % kThreads != 0 && i >= kAllQuads )
                break;
            uint32_t lo[ NS ], hi[ NS ];
            mfmaParts<PREC, NS>( zreg[ r ].x, zreg[ r ].y, lo );
            mfmaParts<PREC, NS>( zreg[ r ].z, zreg[ r ].w, hi );
#pragma unroll
            for ( int q = 0; q < NS; q++ )
                *reinterpret_cast<uint2*>( &sZ[ buf ][ q ][ e * RowH + k ] ) = make_uint2( lo[ q ], hi[ q ] );
        }
        if ( tid < kTile )
            sZn[ slot ][ tid ] = zn;
#pragma unroll
        for ( int r = 0; r < kCLoads; r++ )
        {
            const int i = r * kThreads + tid;
            if ( i < UMAX * kTile )
                sC[ slot ][ ( i % kTile ) * UMAX + i / kTile ] = creg[ r ];
        }
    };

    // Products of one block, in order: group (lvl, t) is step t of the products of order 2^-16, 2^-8, 1
    // (lvl 0, 1, 2; 16-bit modes have the last only), each for P and S.
    constexpr int kLvls = NS == 3 ? 3 : 1, kGroups = kLvls * T;
    constexpr int kProducts = ( NS == 3 ? 12 : 2 ) * T;
    // The next block's products run under this one's exponentials, into a second set of accumulators
    // (one set, and one after the other, where two do not fit the registers, and for the entering
    // pilots' chunks of one or two blocks). At 32 antennas that is so from 13 users on: with two sets
    // 145 registers spilled at 16 users, and 2000 centres took 1474 us for 120k samples, 762 with one (1350
    // before the three-part products).
    constexpr bool PIPE = !SUBTRACT && !MASK && !( NS == 3 && NMAX >= 32 && UMAX > 12 );
    mf32x16 accP[ PIPE ? 2 : 1 ], accS[ PIPE ? 2 : 1 ], accM;
    V az[ 2 ][ NS ];
    auto readGroup = [ & ]( int buf, int cb, auto gC ) {
        constexpr int g = gC, lvl = g / T, t = g % T;
#pragma unroll
        for ( int q = 0; q < kLvls - lvl; q++ )
            az[ g & 1 ][ q ] = *reinterpret_cast<const V*>( &sZ[ buf ][ q ][ ( cb + col ) * RowH + 16 * t + 8 * h ] );
    };
    auto product = [ & ]( int buf, int cb, auto dC, auto kC ) {
        constexpr int d = dC, k = kC;
        constexpr int lvl = NS != 3 || k < 6 * T ? 0 : k < 10 * T ? 1 : 2;
        constexpr int per = NS == 3 ? 6 - 2 * lvl : 2, r = k - ( lvl == 0 ? 0 : lvl == 1 ? 6 * T : 10 * T );
        constexpr int t = r / per, o = r % per / 2, g = lvl * T + t;
        constexpr int pz = o, px = kLvls - 1 - lvl - o; // parts of z and x: their orders add up to the level's
        constexpr int TH = T / 2 > 0 ? T / 2 : 1;
        if constexpr ( r % per == 0 && g + 1 < kGroups )
            readGroup( buf, cb, std::integral_constant<int, ( g + 1 < kGroups ? g + 1 : 0 )> {} );
        const V a = az[ g & 1 ][ pz ];
        const mf32x16 zero {};
        if constexpr ( k % 2 == 0 )
            accP[ d ] = MfmaIn<PREC>::mma( a, xp[ t ][ px ], k == 0 ? zero : accP[ d ] );
        else if constexpr ( HALVES && t >= TH )
            accS[ d ] = MfmaIn<PREC>::mma( a, xp[ t - TH ][ px ], SUBTRACT && lvl == 0 && t == TH && o == 0 ? zero : accS[ d ] );
        else if constexpr ( SUBTRACT )
            accM = MfmaIn<PREC>::mma( a, xp[ t + TH ][ px ], k == 1 ? zero : accM );
        else
            accS[ d ] = MfmaIn<PREC>::mma( a, xs[ t % TX ][ px ], k == 1 ? zero : accS[ d ] );
        if constexpr ( SUBTRACT && k == kProducts - 1 )
            accS[ d ] -= accM;
    };
    // Distances, exponentials and every user's contraction of the block in accumulators S (entries cb of
    // coefficient slot `slot`), between them the products of the next block (entries cbn of buffer
    // bufn) into the other set. The fences keep the two streams interleaved entry by entry.
    // Entries whose coefficients are read ahead together: two where four would spill (32 antennas, two users) or cost the third
    // wave of a SIMD (up to 8 antennas and one user 168 registers instead of 172: 100k samples 61.7 -> 58.5 us).
    constexpr int PF = UMAX > 2 ? 1 : ( UMAX == 2 && NMAX >= 32 ) || ( KEEP && UMAX == 1 && NMAX <= 8 ) ? 2 : 4;
    int run = 0, runLeft = ( nBlocks + ORDER - 1 ) / ORDER; // run of the next phase, blocks left in it
    auto phase = [ & ]( int slot, int cb, int bufn, int cbn, auto dC, auto oC, int rel = 0 ) {
        constexpr int d = dC, ord = oC; // accumulators, sum
        float2 co[ 2 ][ PF * UMAX ];
        float4 zq[ 2 ];
        auto entryOf = [ & ]( int i ) { return cb + 8 * ( i / 4 ) + 4 * h + i % 4; }; // the lane's entry i within the tile
        auto readCo = [ & ]( auto iC ) {
            constexpr int i = iC;
            const float2* cc = &sC[ slot ][ entryOf( i ) * UMAX ];
#pragma unroll
            for ( int u = 0; u < PF * UMAX; u++ )
                co[ i / PF & 1 ][ u ] = cc[ u ];
        };
        if constexpr ( PIPE )
            readGroup( bufn, cbn, std::integral_constant<int, 0> {} );
        zq[ 0 ] = *reinterpret_cast<const float4*>( &sZn[ slot ][ entryOf( 0 ) ] );
        readCo( std::integral_constant<int, 0> {} );
        unrollFor<16>( [ & ]( auto iC ) {
            constexpr int i = iC;
            if constexpr ( i % PF == 0 && i + PF < 16 )
                readCo( std::integral_constant<int, ( i + PF ) % 16> {} );
            if constexpr ( i % 4 == 0 && i + 4 < 16 )
                zq[ ( i / 4 + 1 ) & 1 ] = *reinterpret_cast<const float4*>( &sZn[ slot ][ entryOf( i + 4 ) ] );
            constexpr int k0 = i * kProducts / 16, k1 = ( i + 1 ) * kProducts / 16;
            if constexpr ( PIPE )
                unrollFor<k1 - k0>( [ & ]( auto kC ) { product( bufn, cbn, std::integral_constant<int, 1 - d> {}, std::integral_constant<int, k0 + kC> {} ); } );
            const float4 z4 = zq[ i / 4 & 1 ];
            float q = xq + ( i % 4 == 0 ? z4.x : i % 4 == 1 ? z4.y : i % 4 == 2 ? z4.z : z4.w );
            if constexpr ( MASK ) // arithmetic, as a select of the results costs the scheduler its freedom
                q -= entryOf( i ) >= rel ? 0.f : 1.0e30f;
            const float p = accP[ d ][ i ], s = accS[ d ][ i ];
            // exponentials clamped to 1 (a rounded distance below zero counts as 0)
            const float E0 = __builtin_amdgcn_fmed3f( __builtin_amdgcn_exp2f( fmaf( k2, p, q ) ), 0.f, 1.f );
            const float E1 = __builtin_amdgcn_fmed3f( __builtin_amdgcn_exp2f( fmaf( k2, s, q ) ), 0.f, 1.f );
            const float E2 = __builtin_amdgcn_fmed3f( __builtin_amdgcn_exp2f( fmaf( k2n, s, q ) ), 0.f, 1.f );
#pragma unroll
            for ( int u = 0; u < UMAX; u++ )
            {
                const float2 c = co[ i / PF & 1 ][ i % PF * UMAX + u ];
                fa[ ord ][ u ] = fmaf( c.x, E0, fmaf( c.y, E1, fa[ ord ][ u ] ) );
                fb[ ord ][ u ] = fmaf( c.x, E2, fmaf( c.y, E0, fb[ ord ][ u ] ) );
                asm volatile( "" : "+v"( fa[ ord ][ u ] ), "+v"( fb[ ord ][ u ] )::"memory" );
            }
            __builtin_amdgcn_sched_barrier( 0 );
        } );
        if constexpr ( RUNS )
            if ( --runLeft == 0 ) // the run ends with this block
            {
#pragma unroll
                for ( int u = 0; u < UMAX; u++ )
                {
                    const auto s = __builtin_amdgcn_permlane32_swap( __float_as_uint( fa[ 0 ][ u ] ), __float_as_uint( fb[ 0 ][ u ] ), false, false );
                    ( SUMLDS ? sums[ u * 64 * WAVES ] : sum[ SUMLDS ? 0 : u ] ) += __uint_as_float( s[ 0 ] ) + __uint_as_float( s[ 1 ] );
                    fa[ 0 ][ u ] = fb[ 0 ][ u ] = 0.f;
                }
                run++;
                runLeft = ( nBlocks - run + ORDER - 1 ) / ORDER;
            }
    };

    // Tile tt + 1 is stored between two barriers' reach: its rows (two buffers) replace those of tile
    // tt - 1, last read before the previous barrier, its norms and coefficients (three) those of tile
    // tt - 2, as the last block of a tile is contracted after the barrier.
    constexpr int kBlocks = kTile / 32 / PARTS;
    const int cw = PARTS > 1 ? 32 * ( ( threadIdx.x >> 6 ) % PARTS ) : 0; // the wave's block of a shared-out tile
    typedef std::integral_constant<int, 0> D0;
    const int nTiles = (int)( ( G + kTile - 1 ) / kTile );
    if ( nTiles > 0 )
    {
        loadTile();
        storeTile( 0 );
        if ( nTiles > 1 )
            loadTile();
    }
    __syncthreads();
    auto products = [ & ]( int buf, int cb ) {
        readGroup( buf, cb, D0 {} );
        unrollFor<kProducts>( [ & ]( auto kC ) { product( buf, cb, D0 {}, kC ); } );
    };
    if ( PIPE && nTiles > 0 )
        products( 0, cw );
    auto advance = [ & ]( int tt ) {
        if ( tt + 1 < nTiles )
            storeTile( tt + 1 );
        if ( tt + 2 < nTiles )
            loadTile();
        __syncthreads();
    };
    // (the products past the last block read what the buffers hold, and are not used)
    static_assert( SUMS == 1 || PIPE, "sums kept apart in the pipelined loops" );
    static_assert( SUMS == 1 || kBlocks == 1 || SUMS % kBlocks == 0, "whole turns of the sums" );
    if constexpr ( !PIPE )
    {
#pragma unroll 1
        for ( int tt = 0; tt < nTiles; tt++ )
        {
#pragma unroll 1
            for ( int cb = cw; cb < kTile; cb += 32 * PARTS )
            {
                if ( (int64_t)tt * kTile + cb >= G )
                    break;
                products( tt & 1, cb );
                phase( tt % 3, cb, 0, 0, D0 {}, D0 {}, MASK ? first( (int64_t)tt * kTile ) : 0 );
            }
            advance( tt );
        }
    }
    else if constexpr ( kBlocks == 1 )
    {
        constexpr int STEP = SUMS > 2 ? SUMS : 2;
#pragma unroll 1
        for ( int t0 = 0; t0 < nTiles; t0 += STEP )
            unrollFor<STEP>( [ & ]( auto iC ) {
                const int tt = t0 + iC;
                if ( tt >= nTiles )
                    return;
                advance( tt );
                phase( tt % 3, cw, ( tt + 1 ) & 1, cw, std::integral_constant<int, iC & 1> {}, std::integral_constant<int, iC % SUMS> {} );
            } );
    }
    else
    {
        constexpr int STEP = SUMS > kBlocks ? SUMS / kBlocks : 1;
#pragma unroll 1
        for ( int t0 = 0; t0 < nTiles; t0 += STEP )
            unrollFor<STEP>( [ & ]( auto iC ) {
                const int tt = t0 + iC;
                if ( tt >= nTiles )
                    return;
                unrollFor<kBlocks>( [ & ]( auto bC ) {
                    constexpr int b = bC, last = b == kBlocks - 1;
                    if constexpr ( last )
                        advance( tt );
                    phase( tt % 3, 32 * b, ( tt + last ) & 1, last ? 0 : 32 * b + 32, std::integral_constant<int, b & 1> {},
                           std::integral_constant<int, ( iC * kBlocks + b ) % SUMS> {} );
                } );
            } );
    }
    __syncthreads(); // a following tile stores over what other waves may still read

    if constexpr ( PARTS > 1 )
    {
        const int wave = tid >> 6, part = wave % PARTS;
        addHalves();
        constexpr int kRed = WAVES / PARTS * ( PARTS - 1 ) * UMAX * 64;
        constexpr bool inTile = sizeof( sZ ) >= kRed * sizeof( float2 );
        __shared__ float2 sRed[ inTile ? 1 : kRed ];
        float2* red = ( inTile ? reinterpret_cast<float2*>( sZ ) : sRed ) + wave / PARTS * ( PARTS - 1 ) * UMAX * 64 + lane;
        if ( part > 0 )
#pragma unroll
            for ( int u = 0; u < UMAX; u++ )
                red[ ( ( part - 1 ) * UMAX + u ) * 64 ] = make_float2( fa[ 0 ][ u ], fb[ 0 ][ u ] );
        __syncthreads();
        if ( part == 0 )
        {
#pragma unroll
            for ( int k = 0; k < PARTS - 1; k++ )
#pragma unroll
                for ( int u = 0; u < UMAX; u++ )
                {
                    const float2 v = red[ ( k * UMAX + u ) * 64 ];
                    fa[ 0 ][ u ] += v.x;
                    fb[ 0 ][ u ] += v.y;
                }
            finish( fa[ 0 ], fb[ 0 ] );
        }
        __syncthreads(); // a following tile stores over what was read
    }
    else
    {
        if constexpr ( RUNS )
        {
#pragma unroll
            for ( int u = 0; u < UMAX; u++ )
            {
                fa[ 0 ][ u ] = SUMLDS ? sums[ u * 64 * WAVES ] : sum[ SUMLDS ? 0 : u ];
                fb[ 0 ][ u ] = __shfl_xor( fa[ 0 ][ u ], 32 );
            }
        }
        else
        {
            addHalves();
#pragma unroll
            for ( int o = 1; o < SUMS; o++ )
#pragma unroll
                for ( int u = 0; u < UMAX; u++ )
                {
                    fa[ 0 ][ u ] += fa[ o ][ u ];
                    fb[ 0 ][ u ] += fb[ o ][ u ];
                }
        }
        finish( fa[ 0 ], fb[ 0 ] );
    }
}

// One tile of 32 * WAVES / PARTS data samples of a detect.
template <int NMAX, int UMAX, int PREC, int WAVES = 4, int ETILE = 0, int PARTS = 1>
__device__ __forceinline__ void detectTileMfma( const float* __restrict__ rx, int64_t M, const float* __restrict__ Z,
                                                const float* __restrict__ Zn, const float* __restrict__ C, int64_t ldC,
                                                const float* __restrict__ theta, int64_t G, int U, float wL, float wG, float g2,
                                                float* __restrict__ est, int N, const int64_t tile )
{
    const int h = ( threadIdx.x >> 5 ) & 1;
    const int64_t m = tile * ( 32 * WAVES / PARTS ) + ( threadIdx.x >> 6 ) / PARTS * 32 + ( threadIdx.x & 31 ); // this lane's sample
    const bool valid = m < M;
    const float2* x = reinterpret_cast<const float2*>( rx ) + m;
    constexpr int ORDER = PREC == PREC_F32 && PARTS == 1 ? partsOf( NMAX ) : 1;
    gaussianMfma<NMAX, UMAX, PREC, WAVES, ETILE, false, PARTS, ORDER>(
        Z, Zn, C, ldC, G, U, g2, N, [ & ]( int n ) { return valid && n < N ? x[ (int64_t)n * M ] : make_float2( 0.f, 0.f ); },
        []( int64_t ) { return 0; },
        [ & ]( float( &fa )[ UMAX ], float( &fb )[ UMAX ] ) {
            // f = wL theta . x + wG (Gaussian part), x read again
            if ( !valid || h != 0 )
                return;
            float la[ UMAX ], lb[ UMAX ];
#pragma unroll
            for ( int u = 0; u < UMAX; u++ )
                la[ u ] = lb[ u ] = 0.f;
#pragma unroll 4
            for ( int n = 0; n < N; n++ )
            {
                const float2 v = x[ (int64_t)n * M ];
#pragma unroll
                for ( int u = 0; u < UMAX; u++ )
                {
                    const float* th = theta + ( u < U ? u : 0 ) * 2 * N;
                    la[ u ] += fmaf( th[ n ], v.x, th[ N + n ] * v.y );
                    lb[ u ] += fmaf( th[ n ], v.y, -th[ N + n ] * v.x );
                }
            }
#pragma unroll
            for ( int u = 0; u < UMAX; u++ )
                if ( u < U )
                    reinterpret_cast<float2*>( est )[ (int64_t)u * M + m ] =
                        make_float2( wL * la[ u ] + wG * fa[ u ], wL * lb[ u ] + wG * fb[ u ] );
        } );
}

// Two workgroups of four waves per CU at least: 256 registers per wave, which also keeps the matrix
// results in vector registers (the compiler moves them through accumulation registers otherwise).
template <int NMAX, int UMAX, int PREC>
__global__ void __launch_bounds__( kMfmaThreads, 2 ) apsm_detect_mfma( const float* __restrict__ rx, int64_t M, const float* __restrict__ Z,
                                                                      const float* __restrict__ Zn, const float* __restrict__ C, int64_t ldC,
                                                                      const float* __restrict__ theta, int64_t G, int U, float wL, float wG,
                                                                      float g2, float* __restrict__ est, int N )
{
    detectTileMfma<NMAX, UMAX, PREC>( rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N, blockIdx.x );
}

// Persistent batched detect over a work list (all items of one launch share NMAX and UMAX),
// workgroups of WAVES waves, tiles of 32 * WAVES samples.
template <int NMAX, int UMAX, int PREC, int WAVES = 4, int ETILE = 0>
__global__ void __launch_bounds__( 64 * WAVES, WAVES <= 4 ? 8 / WAVES : 1 ) batch_detect_mfma( const DetDesc* __restrict__ d, const WorkItem* __restrict__ items,
                                                                   int nItems )
{
    for ( int w = blockIdx.x; w < nItems; w += gridDim.x )
    {
        const WorkItem it = items[ w ];
        const DetDesc& x = d[ it.desc ];
        detectTileMfma<NMAX, UMAX, PREC, WAVES, ETILE>( x.rx, x.M, x.Z, x.Zn, x.C, x.ldC, x.theta, x.G, x.U, x.wL, x.wG, x.g2, x.est,
                                                         x.N, it.tile );
    }
}

// Launchers for one precision over every (NMAX, UMAX); each precision's translation unit
// instantiates them.
template <int PREC, int NMAX, int UMAX>
hipError_t launchMfmaNU( hipStream_t s, const float* rx, int64_t M, const float* Z, const float* Zn, const float* C, int64_t ldC,
                         const float* theta, int64_t G, int U, float wL, float wG, float g2, float* est, int N )
{
    hipLaunchKernelGGL( ( apsm_detect_mfma<NMAX, UMAX, PREC> ), dim3( (unsigned)( ( M + kMfmaSamples - 1 ) / kMfmaSamples ) ),
                        dim3( kMfmaThreads ), 0, s, rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N );
    return hipGetLastError();
}

template <int PREC, int NMAX, int UMAX, int WAVES = 4, int ETILE = 0>
hipError_t launchBatchMfmaNU( hipStream_t s, const DetDesc* d, const WorkItem* items, int nItems, int grid )
{
    hipLaunchKernelGGL( ( batch_detect_mfma<NMAX, UMAX, PREC, WAVES, ETILE> ), dim3( grid ), dim3( 64 * WAVES ), 0, s, d, items, nItems );
    return hipGetLastError();
}

// The batched launch in tile shape `shape` (kMfmaShape); shapes other than 0 exist for one-user
// FP32 instances up to 32 antennas (mfmaShapeBuilt).
template <int PREC, int NMAX, int UMAX>
hipError_t launchBatchMfmaShape( int shape, hipStream_t s, const DetDesc* d, const WorkItem* items, int nItems, int grid )
{
    if constexpr ( PREC == PREC_F32 && NMAX <= 32 && UMAX == 1 )
    {
        switch ( shape )
        {
        case 1: return launchBatchMfmaNU<PREC, NMAX, UMAX, 2, 64>( s, d, items, nItems, grid );
        case 2: return launchBatchMfmaNU<PREC, NMAX, UMAX, 4, 32>( s, d, items, nItems, grid );
        case 3: return launchBatchMfmaNU<PREC, NMAX, UMAX, 8, 64>( s, d, items, nItems, grid );
        case 4: return launchBatchMfmaNU<PREC, NMAX, UMAX, 4, 128>( s, d, items, nItems, grid );
        default: break;
        }
    }
    return shape == 0 ? launchBatchMfmaNU<PREC, NMAX, UMAX>( s, d, items, nItems, grid ) : hipErrorInvalidValue;
}

template <int PREC, int NMAX>
struct MfmaTable
{
    template <int UMAX>
    static hipError_t one( bool batch, hipStream_t s, const float* rx, int64_t M, const float* Z, const float* Zn, const float* C,
                           int64_t ldC, const float* theta, int64_t G, int U, float wL, float wG, float g2, float* est, int N,
                           const DetDesc* d, const WorkItem* items, int nItems, int grid, int shape )
    {
        return batch ? launchBatchMfmaShape<PREC, NMAX, UMAX>( shape, s, d, items, nItems, grid )
                     : launchMfmaNU<PREC, NMAX, UMAX>( s, rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N );
    }
    static hipError_t byU( int umax, bool batch, hipStream_t s, const float* rx, int64_t M, const float* Z, const float* Zn,
                           const float* C, int64_t ldC, const float* theta, int64_t G, int U, float wL, float wG, float g2, float* est,
                           int N, const DetDesc* d, const WorkItem* items, int nItems, int grid, int shape )
    {
        switch ( umax )
        {
        case 1: return one<1>( batch, s, rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N, d, items, nItems, grid, shape );
        case 2: return one<2>( batch, s, rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N, d, items, nItems, grid, shape );
        case 4: return one<4>( batch, s, rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N, d, items, nItems, grid, shape );
        case 6: return one<6>( batch, s, rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N, d, items, nItems, grid, shape );
        case 8: return one<8>( batch, s, rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N, d, items, nItems, grid, shape );
        case 10: return one<10>( batch, s, rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N, d, items, nItems, grid, shape );
        case 12: return one<12>( batch, s, rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N, d, items, nItems, grid, shape );
        case 14: return one<14>( batch, s, rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N, d, items, nItems, grid, shape );
        case 16: return one<16>( batch, s, rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N, d, items, nItems, grid, shape );
        default: return hipErrorInvalidValue;
        }
    }
};

template <int PREC>
hipError_t launchMfmaPrec( int nmax, int umax, bool batch, hipStream_t s, const float* rx, int64_t M, const float* Z, const float* Zn,
                           const float* C, int64_t ldC, const float* theta, int64_t G, int U, float wL, float wG, float g2, float* est,
                           int N, const DetDesc* d, const WorkItem* items, int nItems, int grid, int shape )
{
    switch ( nmax )
    {
    case 4: return MfmaTable<PREC, 4>::byU( umax, batch, s, rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N, d, items, nItems, grid, shape );
    case 8: return MfmaTable<PREC, 8>::byU( umax, batch, s, rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N, d, items, nItems, grid, shape );
    case 16: return MfmaTable<PREC, 16>::byU( umax, batch, s, rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N, d, items, nItems, grid, shape );
    case 32: return MfmaTable<PREC, 32>::byU( umax, batch, s, rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N, d, items, nItems, grid, shape );
    case 64: return MfmaTable<PREC, 64>::byU( umax, batch, s, rx, M, Z, Zn, C, ldC, theta, G, U, wL, wG, g2, est, N, d, items, nItems, grid, shape );
    default: return hipErrorInvalidValue;
    }
}

// Entries of each precision's translation unit (defined there).
#define APSM_MFMA_ENTRY( name )                                                                                                   \
    hipError_t name( int nmax, int umax, bool batch, hipStream_t s, const float* rx, int64_t M, const float* Z, const float* Zn,   \
                     const float* C, int64_t ldC, const float* theta, int64_t G, int U, float wL, float wG, float g2, float* est,  \
                     int N, const DetDesc* d, const WorkItem* items, int nItems, int grid, int shape )
APSM_MFMA_ENTRY( mfmaEntryF32 );
APSM_MFMA_ENTRY( mfmaEntryBF16 );
APSM_MFMA_ENTRY( mfmaEntryF16 );

} // namespace apsm
