// Window sequencer of the blocked train path for sampleStep 2 (one complex sample enters per
// step): the projection steps of one block, one workgroup per user, ONE barrier per step.
//
// Per step k the window's rows get beta_k = soft(y - f) / (W (wL|x|^2 + wG)), and every row's f
// grows by the window Gram product G beta_k. The Gram sits in registers: product wave w, lane
// (r, i) = (lane / 16, lane % 16) owns the u-slot v = 16 w + i and the t-slots r TP .. r TP + TP - 1,
// 3 floats per complex pair: A = kappa(a_t,a_v) = kappa(b_t,b_v), C = kappa(b_t,a_v),
// B = kappa(a_t,b_v). So the four partial sums of a row lie in the four 16-lane rows of ONE wave:
// two lane swaps (v_permlane16_swap, v_permlane32_swap) and two adds finish them, with the a-part in
// the lanes of rows 0 and 2 and the b-part in those of rows 1 and 3. f, c, y and the projection weight
// of a slot stay in its lanes' registers from the sample's entry to its departure. The only thing
// that crosses waves is beta, through a double-buffered LDS array: projection k, barrier, product k.
//
// A sample's f needs its share of every earlier coefficient: H_k = P_k + sum_j c_j kappa(j, k). To keep
// that off the chain, a sample takes over its u-slot one step EARLY: after projection k - 1 the slot's
// previous sample leaves (its f is no longer needed, only its beta), the new sample's Gram column is
// loaded into the slot's lanes, and product k - 1 already adds the share of beta_{k-1}. H_k then only
// needs the coefficients after projection k - 2, and helper waves have the whole interval between
// barriers k - 2 and k - 1 to sum it: one takes the window's rows, one the active rows that have
// left the window. P_k is the slot's f from the takeover on (one rounding at its size fewer in every f;
// at TP = 40, where the register it is read ahead into costs 2 %, the first helper adds it). A further helper (the last one, where registers allow only two) streams the
// steps' packages into LDS (global -> LDS DMA, BUFS buffers). The t-slot is taken over at step k itself: the lanes of
// the 16-lane row that holds t-slot p write kappa(p, v) into register p % TP (VGPR index mode).
//
// Bound: the chain LDS write -> barrier -> LDS read -> product -> lane swaps -> projection (about 850
// cycles at the small windows), and vector-ALU issue of the product where several product waves share a
// SIMD (windowSize 160: 160 multiply-adds x 3 waves x 2.2 to 3.1 cycles, of 2500 cycles a step).
// Measured, microseconds per step at windowSize 20 / 40 / 80 / 112 / 160: 0.38 / 0.42 / 0.52 / 0.64 / 1.06;
// with two barriers per step and the projection in waves of its own (as apsm_train_seq2, which still
// runs sampleStep 4) 1.30 / 1.40 / 1.44 / 1.6 / 1.83.
#pragma once

#include "apsm_train2.h"
#include "apsm_win_layout.h"

#include <type_traits>

namespace apsm {

typedef float wf32x4 __attribute__( ( ext_vector_type( 4 ) ) );

// The window Gram of a lane: planes A, C, B of TP floats, read at constant indices, written at a
// wave-uniform one. The compiler writes a vector of 9 to 32 registers in VGPR index mode (a shorter one
// by a select per register, a longer one through memory), so three short planes share one vector
// and at TP = 40 the last 8 registers of each plane are scalars behind a switch.
template <int TP>
struct WinRegs
{
    static constexpr bool ONE = 3 * TP <= 32;
    static constexpr int LO = ONE ? 3 * TP : TP <= 32 ? TP : 32, TAIL = TP > 32 ? TP - 32 : 0;
    typedef float V __attribute__( ( ext_vector_type( LO ) ) );
    V a, c, b; // (ONE: all three planes in a)
    float ta[ TAIL ? TAIL : 1 ], tc[ TAIL ? TAIL : 1 ], tb[ TAIL ? TAIL : 1 ];
    __device__ __forceinline__ float get( int plane, int j ) const
    {
        if ( ONE )
            return a[ plane * TP + j ];
        if ( j < LO )
            return plane == 0 ? a[ j ] : plane == 1 ? c[ j ] : b[ j ];
        return plane == 0 ? ta[ j - LO ] : plane == 1 ? tc[ j - LO ] : tb[ j - LO ];
    }
    __device__ __forceinline__ void put( int plane, int j, float v )
    {
        if ( ONE )
            a[ plane * TP + j ] = v;
        else if ( j < LO )
            ( plane == 0 ? a[ j ] = v : plane == 1 ? c[ j ] = v : b[ j ] = v );
        else
            ( plane == 0 ? ta[ j - LO ] : plane == 1 ? tc[ j - LO ] : tb[ j - LO ] ) = v;
    }
    template <int I>
    __device__ __forceinline__ void insertTail( int j, float xa, float xc, float xb )
    {
        if constexpr ( I < TAIL )
        {
            if ( j == LO + I )
            {
                ta[ I ] = xa;
                tc[ I ] = xc;
                tb[ I ] = xb;
                asm volatile( "" );
            }
            else
                insertTail<I + 1>( j, xa, xc, xb );
        }
    }
    // Slot j (uniform over the wave) of the lanes that take it. The readfirstlane keeps the lane mask a
    // branch: as selects, the writes would copy whole planes.
    __device__ __forceinline__ void insert( int j, bool take, float xa, float xc, float xb )
    {
        if ( take )
        {
            const int js = __builtin_amdgcn_readfirstlane( j );
            if ( TAIL == 0 || js < LO )
            {
                a[ js ] = xa;
                if constexpr ( ONE )
                {
                    a[ TP + js ] = xc;
                    a[ 2 * TP + js ] = xb;
                }
                else
                {
                    c[ js ] = xc;
                    b[ js ] = xb;
                }
            }
            else
                insertTail<0>( js, xa, xc, xb );
        }
    }
};

// The product over this lane's t-slots: fa += A beta_a + C beta_b, fb += B beta_a + A beta_b, the beta pairs
// (q: two t-slots per 16 bytes) read from LDS, one address per 16-lane row, CH pairs of t-slots ahead
// of their multiply-adds. Plain register operands on purpose: two waves of a SIMD then issue a
// multiply-add in 2.2 to 3.1 cycles each (measured), against 4.3 with a DPP or scalar operand, and
// an FP32 matrix instruction shares the vector ALU's multipliers (4 x 4 x 1: 8.2 cycles for two).
template <int TP, typename F>
__device__ __forceinline__ void winProduct( const WinRegs<TP>& g, const float* sBr, float& fa, float& fb, F&& readAhead )
{
    constexpr int Q = ( TP + 1 ) / 2, CH = 2, NCH = ( Q + CH - 1 ) / CH;
    const float4* q4 = reinterpret_cast<const float4*>( sBr );
    float4 q[ 2 ][ CH ];
#pragma unroll
    for ( int m = 0; m < CH; m++ )
        q[ 0 ][ m ] = q4[ m < Q ? m : 0 ];
    readAhead();
    asm volatile( "" ::: "memory" ); // the next step's reads go out here, before the product
    float a0 = 0.f, a1 = 0.f, b0 = 0.f, b1 = 0.f;
#pragma unroll
    for ( int ch = 0; ch < NCH; ch++ )
    {
#pragma unroll
        for ( int m = 0; m < CH; m++ )
            if ( ( ch + 1 ) * CH + m < Q )
                q[ ( ch + 1 ) & 1 ][ m ] = q4[ ( ch + 1 ) * CH + m ];
#pragma unroll
        for ( int m = 0; m < CH; m++ )
        {
            const int j = 2 * ( ch * CH + m );
            const float4 x = q[ ch & 1 ][ m ];
            if ( j < TP )
            {
                a0 = fmaf( x.x, g.get( 0, j ), a0 );
                b0 = fmaf( x.x, g.get( 2, j ), b0 );
                a1 = fmaf( x.y, g.get( 1, j ), a1 );
                b1 = fmaf( x.y, g.get( 0, j ), b1 );
            }
            if ( j + 1 < TP )
            {
                a0 = fmaf( x.z, g.get( 0, j + 1 ), a0 );
                b0 = fmaf( x.z, g.get( 2, j + 1 ), b0 );
                a1 = fmaf( x.w, g.get( 1, j + 1 ), a1 );
                b1 = fmaf( x.w, g.get( 0, j + 1 ), b1 );
            }
        }
        // bound the reads in flight (registers): the next ones stay behind this chunk's multiply-adds
        asm volatile( "" : "+v"( a0 ), "+v"( a1 ), "+v"( b0 ), "+v"( b1 )::"memory" );
    }
    fa = a0 + a1;
    fb = b0 + b1;
}

// Sums of two values over the wave: lanes 0..31 get a's, lanes 32..63 b's.
__device__ __forceinline__ float waveSumPair( float a, float b )
{
    const auto s1 = __builtin_amdgcn_permlane32_swap( __float_as_uint( a ), __float_as_uint( b ), false, false );
    float v = __uint_as_float( s1[ 0 ] ) + __uint_as_float( s1[ 1 ] );
    const auto s2 = __builtin_amdgcn_permlane16_swap( __float_as_uint( v ), __float_as_uint( v ), false, false );
    v = __uint_as_float( s2[ 0 ] ) + __uint_as_float( s2[ 1 ] );
    int x = __float_as_int( v );
    v += __int_as_float( __builtin_amdgcn_update_dpp( 0, x, 0x128, 0xF, 0xF, false ) );
    x = __float_as_int( v );
    v += __int_as_float( __builtin_amdgcn_update_dpp( 0, x, 0x124, 0xF, 0xF, false ) );
    x = __float_as_int( v );
    v += __int_as_float( __builtin_amdgcn_update_dpp( 0, x, 0x4E, 0xF, 0xF, false ) );
    x = __float_as_int( v );
    return v + __int_as_float( __builtin_amdgcn_update_dpp( 0, x, 0xB1, 0xF, 0xF, false ) );
}

// Row indices are relative to the block's first active row a0; Z, Zn point at the first active
// sample, Y and C at the first active real row of user 0 (as in seq2Body). Complex slots follow the
// absolute sample (cMod + rel) % Wc, F is kept by slot [w2].
template <int TP>
__device__ __forceinline__ void winBody( const float* __restrict__ Z, const float* __restrict__ Zn, const float* __restrict__ Y, float* __restrict__ C,
                                         float* __restrict__ Fg, float* __restrict__ thF, const float* __restrict__ P, const float* __restrict__ Gact,
                                         const float* __restrict__ EvF, const Seq2Args& a, const int u )
{
    constexpr int TPQ = winTpq( TP ), PART = winPart( TP ), IMG = winImg( TP ), NP = winProductWaves( TP ), NH = winHelperWaves( TP );
    constexpr int THREADS = winThreads( TP ), BUFS = kWinBufs, VS = 16 * NP, RING = winRing( TP );
    constexpr int PKG = winPkGram( TP ), PKCAP = winPkCap( TP ), NC = PKCAP / 256, SB = winBetaFloats( TP ), RUN = winBetaRun( TP );
    static_assert( VS >= 4 * TP, "a u-slot lane for every slot" );
    static_assert( NC * ( BUFS - 3 ) <= 63, "copies in flight beyond the wait counter" );

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane( tid / 64 );
    const int Wc = a.Wc, w2 = a.w2, K = a.nSteps, newRel0 = a.newRel0, nAct = a.nActC;
    const int cMod = a.a0modW >> 1; // complex slot of relative sample 0
    const int evStride = winEvStride( w2 );

    extern __shared__ float sm[];
    float* sPk = sm; // [BUFS][PKCAP]: image and self entries, eviction shares
    float* sB = sPk + BUFS * PKCAP; // [2][SB]
    float* sCw = sB + 2 * SB; // [2][2 VS]: coefficients of the window after a projection, by slot
    float* sC = sCw + 4 * VS; // [2 kActMax]: coefficients of the active rows that have left the window
    constexpr bool FROZEN = TP < 40; // P_k at the takeover
    // [kActMax + 2][6]: per step the next sample's targets (a, b) and projection weight
    // 1 / (wL|x|^2 + wG), 1 / W of the step itself, and the next sample's frozen shares (a, b)
    float* sStep = sC + 2 * kActMax;
    float* sH = sStep + 6 * ( kActMax + 2 ); // [2][NH][2]: entering shares (window rows, left rows)

    const float* Yu = Y + u * a.ldYC;
    float* Cu = C + u * a.ldYC;
    const float* Pu = P + (int64_t)u * K * 2;
    const float* EvU = EvF + (int64_t)u * K * evStride;

    // package m into buffer slot (one wave; NC copies whatever m is, so that counting waits are
    // constants: past the last step the last package again, without eviction shares stale memory
    // that nothing reads)
    const uint32_t pkLds = __builtin_amdgcn_readfirstlane( (uint32_t)(uintptr_t)( __attribute__( ( address_space( 3 ) ) ) float* )( sPk ) );
    auto pkIssue = [ & ]( int m, int slot ) {
        const int mm = m < K ? m : K - 1;
        const uint32_t dst = pkLds + (uint32_t)( slot * PKCAP ) * 4u;
        const float* src = Gact + winRow( mm, newRel0, Wc, TP );
        const float* ev = EvU + (int64_t)mm * evStride;
#pragma unroll
        for ( int d = 0; d < PKG / 256; d++ )
            dmaDwordx4( src + d * 256, 16u * (uint32_t)lane, __builtin_amdgcn_readfirstlane( dst + (uint32_t)d * 1024u ) );
#pragma unroll
        for ( int d = 0; d < winPkEv( TP ) / 256; d++ )
            dmaDwordx4( ev + d * 256, 16u * (uint32_t)lane, __builtin_amdgcn_readfirstlane( dst + (uint32_t)( PKG + d * 256 ) * 4u ) );
    };
    if ( wave == NP )
        for ( int m = 0; m < BUFS; m++ )
            pkIssue( m, m );

    for ( int i = tid; i < 2 * SB; i += THREADS )
        sB[ i ] = 0.f;
    for ( int i = tid; i < 2 * kActMax; i += THREADS )
        sC[ i ] = 0.f;
    for ( int i = tid; i <= K; i += THREADS ) // record i: step i - 1's next sample is sample i
    {
        const int rel = newRel0 + ( i < K ? i : K - 1 );
        const int W = a.sFirstRel + 2 * i;
        sStep[ 6 * i ] = Yu[ 2 * rel ];
        sStep[ 6 * i + 1 ] = Yu[ 2 * rel + 1 ];
        sStep[ 6 * i + 2 ] = 1.f / ( a.wL * Zn[ rel ] + a.wG );
        sStep[ 6 * i + 3 ] = 1.f / (float)( a.ramp && W < w2 ? W : w2 );
        sStep[ 6 * i + 4 ] = i < K ? Pu[ 2 * i ] : 0.f;
        sStep[ 6 * i + 5 ] = i < K ? Pu[ 2 * i + 1 ] : 0.f;
    }

    const int kLast = newRel0 - 1; // newest sample before the block
    const int pLast = ( cMod + kLast + Wc ) % Wc;

    if ( wave < NP )
    {
        // ================= product waves =================
        const int r = lane >> 4, pt = r & 1, v = wave * 16 + ( lane & 15 );
        const bool vOk = v < Wc;
        int p = pLast + 1 < Wc ? pLast + 1 : 0; // slot of the sample entering at step k
        WinRegs<TP> g;
        float f, c, y, inv;
        {
            int dv = pLast - v;
            dv += dv < 0 ? Wc : 0;
            const int rv = kLast - dv; // sample in this lane's u-slot
            const bool ex = vOk && rv >= 0;
            f = ex ? Fg[ (int64_t)u * w2 + 2 * v + pt ] : 0.f;
            c = ex ? Cu[ 2 * rv + pt ] : 0.f;
            y = ex ? Yu[ 2 * rv + pt ] : 0.f;
            inv = ex ? 1.f / ( a.wL * Zn[ rv ] + a.wG ) : 0.f;
            const float* g0 = Gact + (int64_t)( ex ? v : 0 ) * IMG + r * PART;
            constexpr int VL = TP % 4 == 0 ? 4 : TP % 2 == 0 ? 2 : 1; // floats per load
            typedef float VecL __attribute__( ( ext_vector_type( VL ) ) );
#pragma unroll
            for ( int j = 0; j < TP; j += VL )
            {
                bool ok[ VL ];
#pragma unroll
                for ( int m = 0; m < VL; m++ )
                {
                    const int t = r * TP + j + m;
                    int dt = pLast - t;
                    dt += dt < 0 ? Wc : 0;
                    ok[ m ] = ex && t < Wc && kLast - dt >= 0;
                }
#pragma unroll
                for ( int pl = 0; pl < 3; pl++ )
                {
                    const VecL x = *reinterpret_cast<const VecL*>( g0 + pl * TPQ + j );
#pragma unroll
                    for ( int m = 0; m < VL; m++ )
                    {
                        g.put( pl, j + m, ok[ m ] ? x[ m ] : 0.f );
                    }
                }
                if ( j % 8 >= 8 - VL )
                    __builtin_amdgcn_sched_barrier( 0 );
            }
            if ( lane < 32 )
            {
                sCw[ 2 * VS + 2 * v + pt ] = c;
                sCw[ 2 * v + pt ] = 0.f;
            }
        }
        const int imgV = vOk ? ( v / TP ) * PART + v % TP : 0; // this u-slot's place in an image
        // where this lane's beta goes, and where it reads the ones of its row's t-slots
        float* sBw = sB + 2 * ( v < 4 * TP ? ( v / TP ) * RUN + v % TP : 4 * RUN ) + pt;
        const float* sBr = sB + 2 * r * RUN;
        float* sCv = sCw + 2 * v + pt;
        const int evAt = PKG + ( vOk ? 2 * v + pt : 0 );
        __syncthreads(); // packages 0 .. BUFS - 1 and the LDS arrays are in place
        __syncthreads(); // entering shares of steps 0 and 1
        auto loadColumn = [ & ]( const float* pk ) {
            const float* q = pk + r * PART;
#pragma unroll
            for ( int pl = 0; pl < 3; pl++ )
            {
                if constexpr ( TP % 4 == 0 )
                {
#pragma unroll
                    for ( int j = 0; j < TP / 4; j++ )
                    {
                        const float4 x = reinterpret_cast<const float4*>( q + pl * TPQ )[ j ];
                        g.put( pl, 4 * j, x.x );
                        g.put( pl, 4 * j + 1, x.y );
                        g.put( pl, 4 * j + 2, x.z );
                        g.put( pl, 4 * j + 3, x.w );
                    }
                }
                else
                {
#pragma unroll
                    for ( int j = 0; j < TP; j++ )
                        g.put( pl, j, q[ pl * TPQ + j ] );
                }
            }
        };
        // The entering sample in its u-slot: its kappa with itself (what row insertion needs instead
        // of the image, which there holds the leaving sample)
        float selfA = 0.f, selfC = 0.f;
        bool isP = v == p;
        auto takeOver = [ & ]( const float* pk, float ny, float ninv, float frozen ) {
            f = frozen;
            c = 0.f;
            y = ny;
            inv = ninv;
            selfA = pk[ IMG ];
            selfC = pk[ IMG + 1 ]; // kappa(b,a) = kappa(a,b)
            loadColumn( pk );
        };
        // step 0's sample takes its u-slot over (later ones do so one step early)
        if ( isP )
            takeOver( sPk, sStep[ pt ], sStep[ 2 ], FROZEN ? sStep[ 4 + pt ] : 0.f );
        // read one step ahead: eviction share, kappa(entering, v) for t-slot p, the entering shares,
        // the weight 1 / W, and target and weight of the sample after it
        float evv, rA, rC, rB, h[ NH ], yn, invn, fn = 0.f, iw;
        const float* sRec = sStep; // record of the step read ahead
        auto readAhead = [ & ]( const float* pk, int par ) {
            evv = pk[ evAt ];
            const float* q = pk + imgV;
            rA = q[ 0 ];
            rC = q[ 2 * TPQ ];
            rB = q[ TPQ ];
#pragma unroll
            for ( int i = 0; i < NH; i++ )
                h[ i ] = sH[ ( par * NH + i ) * 2 + pt ];
            iw = sRec[ 3 ];
            yn = sRec[ 6 + pt ];
            invn = sRec[ 8 ];
            if ( FROZEN )
                fn = sRec[ 10 + pt ];
            sRec += 6;
        };
        readAhead( sPk, 0 );
        float x = 0.f; // this row's product of the previous step
        int rp = p / TP, jp = p - rp * TP; // 16-lane row and register of t-slot p
        const int rSel = vOk ? r : -1;
        int slot = 0; // k % BUFS
        int relOld = newRel0 + 1 - Wc; // sample that leaves after step k's projection

        auto step = [ & ]( auto half ) { // k & 1
            const int pn = p + 1 < Wc ? p + 1 : 0;
            slot = ( slot + 1 ) & ( BUFS - 1 );
            const float* pkn = sPk + slot * PKCAP;
            // ---- projection ----
            float hs = h[ 0 ] + h[ 1 ];
            if constexpr ( NH > 2 )
                hs += h[ 2 ];
            // (one rounding at f's size: the shares are added up among themselves first)
            f += x + ( ( isP ? hs : 0.f ) - ( a.hasEv ? evv : 0.f ) );
            const float res = y - f;
            // (for a residual that is not a number, an unknown target's, maximum and minimum give the other
            // operand: it projects nothing)
            const float bb = fmaxf( res, a.eB ) + fminf( res, -a.eB );
            const float beta = bb * ( iw * inv );
            c += beta;
            // (the two upper rows of a wave write what the two lower ones write)
            sBw[ half * SB ] = beta;
            sCv[ half * 2 * VS ] = c;
            const bool leave = v == pn;
            if ( leave )
            {
                sCv[ half * 2 * VS ] = 0.f;
                if ( relOld >= 0 )
                    sC[ 2 * relOld + pt ] = c;
            }
            relOld++;
            // ---- t-slot p: the sample that enters now ----
            g.insert( jp, rSel == rp, isP ? selfA : rA, isP ? selfC : rC, isP ? selfC : rB );
            asm volatile( "s_waitcnt lgkmcnt(0)" ::: "memory" );
            // ---- u-slot pn: the sample of the next step (the reads need not end before the barrier;
            //      after the last step it takes a stale package, whose slot nothing reads) ----
            if ( leave )
                takeOver( pkn, yn, invn, FROZEN ? fn : 0.f );
            isP = leave;
            asm volatile( "s_barrier" ::: "memory" );
            // ---- product, with the next step's reads in flight ----
            float fa, fb;
            winProduct<TP>( g, sBr + half * SB, fa, fb, [ & ] { readAhead( pkn, half ^ 1 ); } );
            // rows 0 and 2 of the wave take the a-part, rows 1 and 3 the b-part
            const auto s1 = __builtin_amdgcn_permlane16_swap( __float_as_uint( fa ), __float_as_uint( fb ), false, false );
            const float xh = __uint_as_float( s1[ 0 ] ) + __uint_as_float( s1[ 1 ] );
            const auto s2 = __builtin_amdgcn_permlane32_swap( __float_as_uint( xh ), __float_as_uint( xh ), false, false );
            x = __uint_as_float( s2[ 0 ] ) + __uint_as_float( s2[ 1 ] );
            // (the reads ahead are not moved behind the product)
            asm volatile( "" : "+v"( evv ), "+v"( rA ), "+v"( rC ), "+v"( rB ), "+v"( h[ 0 ] ), "+v"( h[ 1 ] ), "+v"( yn ), "+v"( invn ), "+v"( iw ) );
            if ( FROZEN )
                asm volatile( "" : "+v"( fn ) );
            p = pn;
            jp++;
            if ( jp == TP || p == 0 )
            {
                jp = 0;
                rp = p == 0 ? 0 : rp + 1;
            }
        };
        if constexpr ( TP == 40 ) // (unrolled by two, the loop does not fit the registers)
#pragma unroll 1
            for ( int k = 0; k < K; k++ )
                step( k & 1 );
        else
#pragma unroll 1
            for ( int k = 0; k < K; k += 2 )
            {
                step( std::integral_constant<int, 0> {} );
                if ( k + 1 < K )
                    step( std::integral_constant<int, 1> {} );
            }
        f += x;
        if ( lane < 32 && vOk )
        {
            Fg[ (int64_t)u * w2 + 2 * v + pt ] = f;
            const int kEnd = newRel0 + K - 1;
            int dv = ( p > 0 ? p - 1 : Wc - 1 ) - v;
            dv += dv < 0 ? Wc : 0;
            if ( kEnd - dv >= 0 && !isP ) // (slot p has been taken over; its sample's c is in sC already)
                sC[ 2 * ( kEnd - dv ) + pt ] = c;
        }
    }
    else
    {
        // ================= helper waves =================
        // Interval k (after barrier k): the packages' wave issues package k + BUFS into the buffer step k
        // released; the entering share H_{k+2} is summed.
        // window rows in H_m, coefficients as after projection m - 2 (buffer cw)
        int tOff[ ( 4 * TP + 63 ) / 64 ];
#pragma unroll
        for ( int i = 0; i < ( 4 * TP + 63 ) / 64; i++ )
        {
            const int t = i * 64 + lane < 4 * TP ? i * 64 + lane : 4 * TP - 1;
            tOff[ i ] = ( t / TP ) * PART + t % TP;
        }
        auto windowShare = [ & ]( int m, int cw ) {
            const float* pk = sPk + ( m & ( BUFS - 1 ) ) * PKCAP;
            const float2* cs = reinterpret_cast<const float2*>( sCw + cw * 2 * VS );
            float ea = 0.f, eb = 0.f;
#pragma unroll
            for ( int i = 0; i < ( 4 * TP + 63 ) / 64; i++ )
            {
                const bool ok = i * 64 + lane < 4 * TP;
                const float* q = pk + tOff[ i ];
                const float2 cc = cs[ ok ? i * 64 + lane : 0 ];
                const float A = q[ 0 ], Cq = q[ TPQ ], Bq = q[ 2 * TPQ ];
                const float sa = cc.x * A + cc.y * Cq, sb = cc.x * Bq + cc.y * A;
                ea += ok ? sa : 0.f;
                eb += ok ? sb : 0.f;
            }
            const float s = waveSumPair( ea, eb );
            if ( ( lane & 31 ) == 0 )
                sH[ ( m & 1 ) * NH * 2 + ( lane >> 5 ) ] = FROZEN ? s : s + sStep[ 6 * m + 4 + ( lane >> 5 ) ];
        };
        // the active rows that have left the window by step m - 1 (LEFT * 256 of them from `base` on);
        // their kappa planes come from memory through a ring of register sets
        constexpr int LEFT = kActMax / 256 / ( NH - 1 );
        struct Left
        {
            wf32x4 A[ LEFT ], B[ LEFT ], C[ LEFT ];
        };
        auto leftLoad = [ & ]( int m, int base, Left& q ) {
            const int mm = m < K ? m : K - 1;
            const int o4 = ( winOlder( mm, newRel0, Wc ) + 3 ) & ~3;
            const float* src = Gact + winRow( mm, newRel0, Wc, TP ) + IMG + 4;
#pragma unroll
            for ( int i = 0; i < LEFT; i++ )
            {
                const int jj = base + i * 256 + 4 * lane;
                const int j = jj < o4 ? jj : 0; // (row 0: never past the buffer)
                q.A[ i ] = *reinterpret_cast<const wf32x4*>( src + j );
                q.B[ i ] = *reinterpret_cast<const wf32x4*>( src + o4 + j );
                q.C[ i ] = *reinterpret_cast<const wf32x4*>( src + 2 * o4 + j );
            }
        };
        auto leftShare = [ & ]( int m, int base, int src, const Left& q ) {
            const int older = winOlder( m, newRel0, Wc );
            float ea = 0.f, eb = 0.f;
#pragma unroll
            for ( int i = 0; i < LEFT; i++ )
            {
                const int j = base + i * 256 + 4 * lane;
                const float4 c0 = *reinterpret_cast<const float4*>( sC + 2 * j ), c1 = *reinterpret_cast<const float4*>( sC + 2 * j + 4 );
                const wf32x4 A = q.A[ i ], B = q.B[ i ], Cq = q.C[ i ];
                float sa = c0.x * A[ 0 ] + c0.y * B[ 0 ] + c0.z * A[ 1 ] + c0.w * B[ 1 ];
                float sb = c0.x * Cq[ 0 ] + c0.y * A[ 0 ] + c0.z * Cq[ 1 ] + c0.w * A[ 1 ];
                sa += c1.x * A[ 2 ] + c1.y * B[ 2 ] + c1.z * A[ 3 ] + c1.w * B[ 3 ];
                sb += c1.x * Cq[ 2 ] + c1.y * A[ 2 ] + c1.z * Cq[ 3 ] + c1.w * A[ 3 ];
                ea += j < older ? sa : 0.f;
                eb += j < older ? sb : 0.f;
            }
            const float s = waveSumPair( ea, eb );
            if ( ( lane & 31 ) == 0 )
                sH[ ( ( m & 1 ) * NH + src ) * 2 + ( lane >> 5 ) ] = s;
        };
        const int role = wave - NP; // 0: packages and window rows, others: left rows
        if ( role > 0 )
        {
            const int base = ( role - 1 ) * 256;
            Left ring[ RING ]; // set m % RING: step m
            Left first;
            leftLoad( 0, base, first );
            leftLoad( 1, base, ring[ 1 % RING ] );
#pragma unroll
            for ( int m = 2; m < RING + 1; m++ )
                leftLoad( m, base, m == RING ? ring[ 0 ] : ring[ m ] );
            __syncthreads();
            leftShare( 0, base, role, first );
            if ( K > 1 )
                leftShare( 1, base, role, ring[ 1 ] );
            leftLoad( RING + 1, base, ring[ 1 ] );
            __syncthreads();
#pragma unroll 1
            for ( int k0 = 0; k0 < K; k0 += RING )
            {
#pragma unroll
                for ( int d = 0; d < RING; d++ )
                {
                    const int k = k0 + d;
                    if ( k >= K )
                        break;
                    ldsBarrier();
                    if ( k + 2 < K )
                        leftShare( k + 2, base, role, ring[ ( d + 2 ) % RING ] );
                    leftLoad( k + 2 + RING, base, ring[ ( d + 2 ) % RING ] );
                }
            }
        }
        else
        {
            waitVm<0>();
            __syncthreads();
            for ( int m = 0; m < 2 && m < K; m++ )
                windowShare( m, 1 );
            __syncthreads();
#pragma unroll 1
            for ( int k = 0; k < K; k++ )
            {
                ldsBarrier();
                pkIssue( k + BUFS, k & ( BUFS - 1 ) );
                if ( k + 2 < K )
                    windowShare( k + 2, k & 1 );
                // package k + 3 is first read after the next barrier; the younger ones stay in flight
                waitVm<NC*( BUFS - 3 )>();
            }
            waitVm<0>(); // the buffers are reused below
        }
    }
    __syncthreads();

    // write back c of the active rows; thF += c_j x_j of the rows leaving the active set
    for ( int i = tid; i < 2 * nAct; i += THREADS )
        Cu[ i ] = sC[ i ];
    const int N = a.N, L = a.L, chunks = THREADS / N;
    float* red = sPk; // [chunks][L]
    {
        const int d = tid % N, ch = tid / N;
        if ( ch < chunks )
        {
            float re = 0.f, im = 0.f;
#pragma unroll 8
            for ( int j = ch; j < a.nFr; j += chunks )
            {
                const float* zj = Z + (int64_t)j * L + d;
                const float zr = zj[ 0 ], zi = zj[ N ];
                const float2 cc = *reinterpret_cast<const float2*>( sC + 2 * j );
                re += cc.x * zr + cc.y * zi;
                im += cc.x * zi - cc.y * zr;
            }
            red[ ch * L + d ] = re;
            red[ ch * L + N + d ] = im;
        }
    }
    __syncthreads();
    if ( tid < L )
    {
        // In FP64, one rounding per block: every later sample's frozen share has this sum's error, and
        // added up in FP32 (32 to 320 roundings a block) it made most of a trained detector's error: 16
        // antennas, 10 users, windowSize 160, 700 pilots: estimates off by 3.0e-7 rms of their own, 1.3e-7 now.
        double acc = thF[ u * L + tid ];
        for ( int ch = 0; ch < chunks; ch++ )
            acc += red[ ch * L + tid ];
        thF[ u * L + tid ] = (float)acc;
    }
}

template <int TP>
__global__ void __launch_bounds__( winThreads( TP ) ) apsm_train_win( const float* __restrict__ Z, const float* __restrict__ Zn, const float* __restrict__ Y,
                                                                     float* __restrict__ C, float* __restrict__ Fg, float* __restrict__ thF,
                                                                     const float* __restrict__ P, const float* __restrict__ Gact,
                                                                     const float* __restrict__ EvF, const Seq2Args a )
{
    winBody<TP>( Z, Zn, Y, C, Fg, thF, P, Gact, EvF, a, blockIdx.x );
}

} // namespace apsm
