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
// A wave reads its beta pairs once per lane (ceil(TP / 16) 8-byte LDS reads) and broadcasts each
// inside the 16-lane row by DPP (row_newbcast) in the multiply-adds themselves.
//
// A sample's f needs its share of every earlier coefficient: H_k = P_k + sum_j c_j kappa(j, k). To keep
// that off the chain, a sample takes over its u-slot one step EARLY: after projection k - 1 the slot's
// previous sample leaves (its f is no longer needed, only its beta), the new sample's Gram column is
// loaded into the slot's lanes, and product k - 1 already adds the share of beta_{k-1}. H_k then only
// needs the coefficients after projection k - 2, and helper waves have the whole interval between
// barriers k - 2 and k - 1 to sum it: one takes the window's rows and P_k, one the active rows that have
// left the window. A further helper (the last one, where registers allow only two) streams the
// steps' packages into LDS (global -> LDS DMA, BUFS buffers). The t-slot is taken over at step k itself: the lanes of
// the 16-lane row that holds t-slot p write kappa(p, v) into register p % TP (VGPR index mode).
//
// Bound: vector-ALU issue of the product where several product waves share a SIMD (windowSize 160:
// 160 multiply-adds x 3 waves x 4 cycles = 1920 of the step's cycles), below that the chain LDS
// write -> barrier -> LDS read -> product -> lane swaps -> projection.
#pragma once

#include "apsm_train2.h"
#include "apsm_win_layout.h"

namespace apsm {

// s_waitcnt vmcnt(min(n, 31)) for a wave-uniform n
__device__ __forceinline__ void waitVmUpTo31( int n )
{
    switch ( n )
    {
    case 16: waitVm<16>(); break;
    case 17: waitVm<17>(); break;
    case 18: waitVm<18>(); break;
    case 19: waitVm<19>(); break;
    case 20: waitVm<20>(); break;
    case 21: waitVm<21>(); break;
    case 22: waitVm<22>(); break;
    case 23: waitVm<23>(); break;
    case 24: waitVm<24>(); break;
    case 25: waitVm<25>(); break;
    case 26: waitVm<26>(); break;
    case 27: waitVm<27>(); break;
    case 28: waitVm<28>(); break;
    case 29: waitVm<29>(); break;
    case 30: waitVm<30>(); break;
    default:
        if ( n > 30 )
            waitVm<31>();
        else
            waitVmN( n );
        break;
    }
}

// One register plane of the window Gram: TP floats, read at constant indices, written at a
// wave-uniform one (VGPR index mode works on up to 32 registers, so TP = 40 is 32 + 8).
template <int TP>
struct WinPlane
{
    static constexpr int LO = TP <= 32 ? TP : 32, HI = TP <= 32 ? 2 : TP - 32;
    typedef float VLo __attribute__( ( ext_vector_type( LO ) ) );
    typedef float VHi __attribute__( ( ext_vector_type( HI ) ) );
    VLo lo;
    VHi hi;
    __device__ __forceinline__ float get( int j ) const { return j < LO ? lo[ j ] : hi[ j - LO ]; }
    __device__ __forceinline__ void put( int j, float v ) // constant j
    {
        if ( j < LO )
            lo[ j ] = v;
        else
            hi[ j - LO ] = v;
    }
};

// Four t-slots I .. I + 3 of the product: acc += kappa * beta with the beta pair of t-slot I + m taken
// from lane I + m of the 16-lane row. The leading s_nop gives a preceding vector write of the
// beta registers (a copy the compiler may place) its two wait states before the DPP reads.
template <int I>
__device__ __forceinline__ void winFma4( float& a0, float& b0, float& a1, float& b1, const float bx, const float by, const float A0, const float A1,
                                         const float A2, const float A3, const float C0, const float C1, const float C2, const float C3,
                                         const float B0, const float B1, const float B2, const float B3 )
{
#define APSM_WF( acc, bt, g, i ) "v_fmac_f32_dpp " acc ", " bt ", " g " row_newbcast:" i " row_mask:0xf bank_mask:0xf\n\t"
    asm( "s_nop 1\n\t" APSM_WF( "%0", "%4", "%6", "%18" ) APSM_WF( "%1", "%5", "%6", "%18" ) APSM_WF( "%2", "%5", "%10", "%18" )
             APSM_WF( "%3", "%4", "%14", "%18" ) APSM_WF( "%0", "%4", "%7", "%19" ) APSM_WF( "%1", "%5", "%7", "%19" )
                 APSM_WF( "%2", "%5", "%11", "%19" ) APSM_WF( "%3", "%4", "%15", "%19" ) APSM_WF( "%0", "%4", "%8", "%20" )
                     APSM_WF( "%1", "%5", "%8", "%20" ) APSM_WF( "%2", "%5", "%12", "%20" ) APSM_WF( "%3", "%4", "%16", "%20" )
                         APSM_WF( "%0", "%4", "%9", "%21" ) APSM_WF( "%1", "%5", "%9", "%21" ) APSM_WF( "%2", "%5", "%13", "%21" )
                             APSM_WF( "%3", "%4", "%17", "%21" )
         : "+v"( a0 ), "+v"( b0 ), "+v"( a1 ), "+v"( b1 )
         : "v"( bx ), "v"( by ), "v"( A0 ), "v"( A1 ), "v"( A2 ), "v"( A3 ), "v"( C0 ), "v"( C1 ), "v"( C2 ), "v"( C3 ), "v"( B0 ), "v"( B1 ),
           "v"( B2 ), "v"( B3 ), "n"( I ), "n"( I + 1 ), "n"( I + 2 ), "n"( I + 3 ) );
}
template <int I>
__device__ __forceinline__ void winFma1( float& a0, float& b0, float& a1, float& b1, const float bx, const float by, const float A, const float C, const float B )
{
    asm( "s_nop 1\n\t" APSM_WF( "%0", "%4", "%6", "%9" ) APSM_WF( "%1", "%5", "%6", "%9" ) APSM_WF( "%2", "%5", "%7", "%9" )
             APSM_WF( "%3", "%4", "%8", "%9" )
         : "+v"( a0 ), "+v"( b0 ), "+v"( a1 ), "+v"( b1 )
         : "v"( bx ), "v"( by ), "v"( A ), "v"( C ), "v"( B ), "n"( I ) );
#undef APSM_WF
}

// The product over t-slots J .. TP - 1 of this lane's part; beta pairs of t-slot j in bt[j / 16].
template <int TP, int J>
__device__ __forceinline__ void winProduct( float& a0, float& b0, float& a1, float& b1, const float2* bt, const WinPlane<TP>& gA,
                                            const WinPlane<TP>& gC, const WinPlane<TP>& gB )
{
    if constexpr ( J + 4 <= TP && J % 16 <= 12 )
    {
        winFma4<J % 16>( a0, b0, a1, b1, bt[ J / 16 ].x, bt[ J / 16 ].y, gA.get( J ), gA.get( J + 1 ), gA.get( J + 2 ), gA.get( J + 3 ), gC.get( J ),
                         gC.get( J + 1 ), gC.get( J + 2 ), gC.get( J + 3 ), gB.get( J ), gB.get( J + 1 ), gB.get( J + 2 ), gB.get( J + 3 ) );
        winProduct<TP, J + 4>( a0, b0, a1, b1, bt, gA, gC, gB );
    }
    else if constexpr ( J < TP )
    {
        winFma1<J % 16>( a0, b0, a1, b1, bt[ J / 16 ].x, bt[ J / 16 ].y, gA.get( J ), gC.get( J ), gB.get( J ) );
        winProduct<TP, J + 1>( a0, b0, a1, b1, bt, gA, gC, gB );
    }
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
    constexpr int THREADS = winThreads( TP ), BUFS = winBufs( TP ), MB = ( TP + 15 ) / 16, VS = 16 * NP;
    constexpr int PKG = winPkGram( TP ), PKCAP = winPkCap( TP ), SB = winBetaFloats( TP );
    static_assert( VS >= 4 * TP, "a u-slot lane for every slot" );

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane( tid / 64 );
    const int Wc = a.Wc, w2 = a.w2, K = a.nSteps, newRel0 = a.newRel0, nAct = a.nActC;
    const int cMod = a.a0modW >> 1; // complex slot of relative sample 0
    const int evStride = winEvStride( w2 );

    extern __shared__ float sm[];
    float* sPk = sm; // [BUFS][PKCAP]: Gram part, eviction shares
    float* sB = sPk + BUFS * PKCAP; // [2][SB]
    float* sCw = sB + 2 * SB; // [2][2 VS]: coefficients of the window after a projection, by slot
    float* sC = sCw + 4 * VS; // [2 kActMax]: coefficients of the active rows that have left the window
    float* sY = sC + 2 * kActMax; // [2 K]: targets, projection weights and frozen shares of the entering samples
    float* sInv = sY + 2 * kActMax; // [K]
    float* sP = sInv + kActMax; // [2 K]
    float* sH = sP + 2 * kActMax; // [2][4]: entering shares (window + P: a, b; left rows: a, b)

    const float* Yu = Y + u * a.ldYC;
    float* Cu = C + u * a.ldYC;
    const float* Pu = P + (int64_t)u * K * 2;
    const float* EvU = EvF + (int64_t)u * K * evStride;

    // ---- packages (one wave) ----
    const uint32_t pkLds = __builtin_amdgcn_readfirstlane( (uint32_t)(uintptr_t)( __attribute__( ( address_space( 3 ) ) ) float* )( sPk ) );
    const int nE = a.hasEv ? ( evStride + 255 ) / 256 : 0;
    auto pkCopies = [ & ]( int m ) { return ( IMG + 4 + 3 * ( ( winOlder( m, newRel0, Wc ) + 3 ) & ~3 ) + 255 ) / 256 + nE; };
    auto pkIssue = [ & ]( int m ) {
        const uint32_t dst = pkLds + (uint32_t)( ( m % BUFS ) * PKCAP ) * 4u;
        const float* src = Gact + winRow( m, newRel0, Wc, TP );
        const int nG = pkCopies( m ) - nE;
#pragma unroll 1
        for ( int d = 0; d < nG; d++ )
            dmaDwordx4( src + d * 256, 16u * (uint32_t)lane, __builtin_amdgcn_readfirstlane( dst + (uint32_t)d * 1024u ) );
        const float* ev = EvU + (int64_t)m * evStride;
#pragma unroll 1
        for ( int d = 0; d < nE; d++ )
            dmaDwordx4( ev + d * 256, 16u * (uint32_t)lane, __builtin_amdgcn_readfirstlane( dst + (uint32_t)( PKG + d * 256 ) * 4u ) );
    };
    if ( wave == NP )
        for ( int m = 0; m < BUFS && m < K; m++ )
            pkIssue( m );

    for ( int i = tid; i < 2 * SB; i += THREADS )
        sB[ i ] = 0.f;
    for ( int i = tid; i < 2 * kActMax; i += THREADS )
        sC[ i ] = 0.f;
    for ( int i = tid; i < 2 * K; i += THREADS )
    {
        sY[ i ] = Yu[ 2 * newRel0 + i ];
        sP[ i ] = Pu[ i ];
    }
    for ( int i = tid; i < K; i += THREADS )
        sInv[ i ] = 1.f / ( a.wL * Zn[ newRel0 + i ] + a.wG );

    const int kLast = newRel0 - 1; // newest sample before the block
    const int pLast = ( cMod + kLast + Wc ) % Wc;
    int p = pLast + 1 < Wc ? pLast + 1 : 0; // slot of the sample entering at step k
    const float invWfull = 1.f / (float)w2;

    if ( wave < NP )
    {
        // ================= product waves =================
        const int r = lane >> 4, pt = r & 1, v = wave * 16 + ( lane & 15 );
        const bool vOk = v < Wc;
        WinPlane<TP> gA, gC, gB;
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
#pragma unroll
            for ( int j = 0; j < TP; j++ )
            {
                const int t = r * TP + j;
                int dt = pLast - t;
                dt += dt < 0 ? Wc : 0;
                const bool ok = ex && t < Wc && kLast - dt >= 0;
                const float xa = g0[ j ], xc = g0[ TPQ + j ], xb = g0[ 2 * TPQ + j ];
                gA.put( j, ok ? xa : 0.f );
                gC.put( j, ok ? xc : 0.f );
                gB.put( j, ok ? xb : 0.f );
                if ( ( j & 7 ) == 7 )
                    __builtin_amdgcn_sched_barrier( 0 );
            }
            if ( lane < 32 )
            {
                sCw[ 2 * VS + 2 * v + pt ] = c;
                sCw[ 2 * v + pt ] = 0.f;
            }
        }
        const int imgV = ( v / TP ) * PART + v % TP; // this u-slot's place in an image
        __syncthreads(); // packages 0 .. BUFS - 1 and the LDS arrays are in place
        __syncthreads(); // entering shares of steps 0 and 1
        auto loadColumn = [ & ]( const float* pk ) {
            const float* q = pk + r * PART;
            if constexpr ( TP % 4 == 0 )
            {
                const float4* q4 = reinterpret_cast<const float4*>( q );
#pragma unroll
                for ( int j = 0; j < TP / 4; j++ )
                {
                    const float4 xa = q4[ j ], xc = q4[ TPQ / 4 + j ], xb = q4[ TPQ / 2 + j ];
                    const float va[ 4 ] = { xa.x, xa.y, xa.z, xa.w }, vc[ 4 ] = { xc.x, xc.y, xc.z, xc.w }, vb[ 4 ] = { xb.x, xb.y, xb.z, xb.w };
#pragma unroll
                    for ( int m = 0; m < 4; m++ )
                    {
                        gA.put( 4 * j + m, va[ m ] );
                        gC.put( 4 * j + m, vc[ m ] );
                        gB.put( 4 * j + m, vb[ m ] );
                    }
                }
            }
            else
            {
#pragma unroll
                for ( int j = 0; j < TP; j++ )
                {
                    gA.put( j, q[ j ] );
                    gC.put( j, q[ TPQ + j ] );
                    gB.put( j, q[ 2 * TPQ + j ] );
                }
            }
        };
        // step 0's sample takes its u-slot over (later ones do so one step early)
        if ( v == p )
        {
            f = 0.f;
            c = 0.f;
            y = sY[ pt ];
            inv = sInv[ 0 ];
            loadColumn( sPk );
        }
        float x = 0.f; // this row's product of the previous step
        float evv = a.hasEv ? sPk[ PKG + ( vOk ? 2 * v + pt : 0 ) ] : 0.f;
        float h = v == p ? sH[ pt ] + sH[ 2 + pt ] : 0.f;
        float rA, rC, rB; // kappa(entering, v): what t-slot p gets
        {
            const bool self = v == p;
            const int o = self ? IMG : ( vOk ? imgV : 0 ), st = self ? 1 : TPQ;
            rA = sPk[ o ];
            rC = sPk[ o + ( self ? 1 : 2 * TPQ ) ];
            rB = sPk[ o + ( self ? 2 : st ) ];
        }
        float yn = K > 1 ? sY[ 2 + pt ] : 0.f, invn = K > 1 ? sInv[ 1 ] : 0.f;
        int rp = p / TP, jp = p - rp * TP; // 16-lane row and register of t-slot p

#pragma unroll 1
        for ( int k = 0; k < K; k++ )
        {
            const bool more = k + 1 < K;
            const int pn = p + 1 < Wc ? p + 1 : 0;
            // ---- projection ----
            if ( a.hasEv )
                f -= evv;
            f += x + h;
            const float res = y - f;
            const float bb = res - __builtin_amdgcn_fmed3f( res, -a.eB, a.eB );
            float invW = invWfull;
            if ( a.ramp )
            {
                const int W = a.sFirstRel + 2 * k;
                invW = 1.f / (float)( W < w2 ? W : w2 );
            }
            const float beta = bb * invW * inv;
            c += beta;
            const bool leave = more && v == pn;
            if ( lane < 32 )
            {
                sB[ ( k & 1 ) * SB + 2 * v + pt ] = beta;
                sCw[ ( k & 1 ) * 2 * VS + 2 * v + pt ] = leave ? 0.f : c;
                const int relOld = newRel0 + k + 1 - Wc; // sample leaving slot pn
                if ( leave && relOld >= 0 )
                    sC[ 2 * relOld + pt ] = c;
            }
            // ---- t-slot p: the sample that enters now ----
            if ( r == rp && vOk )
            {
                // the active lanes share r, so jp is uniform: one indexed register write per plane
                const int js = __builtin_amdgcn_readfirstlane( jp );
                if ( TP <= 32 || js < 32 )
                {
                    gA.lo[ js ] = rA;
                    gC.lo[ js ] = rC;
                    gB.lo[ js ] = rB;
                }
                else
                {
                    gA.hi[ js - 32 ] = rA;
                    gC.hi[ js - 32 ] = rC;
                    gB.hi[ js - 32 ] = rB;
                }
            }
            // ---- u-slot pn: the sample of the next step ----
            const float* pkn = sPk + ( ( k + 1 ) % BUFS ) * PKCAP;
            if ( leave )
            {
                f = 0.f;
                c = 0.f;
                y = yn;
                inv = invn;
                loadColumn( pkn );
            }
            ldsBarrier();
            // ---- product, with the next step's reads in flight ----
            float2 bt[ MB ];
            const float2* sB2 = reinterpret_cast<const float2*>( sB + ( k & 1 ) * SB ) + r * TP + ( lane & 15 );
#pragma unroll
            for ( int m = 0; m < MB; m++ )
                bt[ m ] = sB2[ 16 * m ];
            h = 0.f;
            if ( more )
            {
                if ( a.hasEv )
                    evv = pkn[ PKG + ( vOk ? 2 * v + pt : 0 ) ];
                const bool self = v == pn;
                const int o = self ? IMG : ( vOk ? imgV : 0 );
                rA = pkn[ o ];
                rC = pkn[ o + ( self ? 1 : 2 * TPQ ) ];
                rB = pkn[ o + ( self ? 2 : TPQ ) ];
                if ( self )
                    h = sH[ ( ( k + 1 ) & 1 ) * 4 + pt ] + sH[ ( ( k + 1 ) & 1 ) * 4 + 2 + pt ];
                if ( k + 2 < K )
                {
                    yn = sY[ 2 * ( k + 2 ) + pt ];
                    invn = sInv[ k + 2 ];
                }
            }
            float a0 = 0.f, b0 = 0.f, a1 = 0.f, b1 = 0.f;
            winProduct<TP, 0>( a0, b0, a1, b1, bt, gA, gC, gB );
            // rows 0 and 2 of the wave take the a-part, rows 1 and 3 the b-part
            const auto s1 = __builtin_amdgcn_permlane16_swap( __float_as_uint( a0 + a1 ), __float_as_uint( b0 + b1 ), false, false );
            const float xh = __uint_as_float( s1[ 0 ] ) + __uint_as_float( s1[ 1 ] );
            const auto s2 = __builtin_amdgcn_permlane32_swap( __float_as_uint( xh ), __float_as_uint( xh ), false, false );
            x = __uint_as_float( s2[ 0 ] ) + __uint_as_float( s2[ 1 ] );
            p = pn;
            jp++;
            if ( jp == TP || p == 0 )
            {
                jp = 0;
                rp = p == 0 ? 0 : rp + 1;
            }
        }
        f += x;
        if ( lane < 32 && vOk )
        {
            Fg[ (int64_t)u * w2 + 2 * v + pt ] = f;
            const int kEnd = newRel0 + K - 1;
            int dv = ( p > 0 ? p - 1 : Wc - 1 ) - v;
            dv += dv < 0 ? Wc : 0;
            if ( kEnd - dv >= 0 )
                sC[ 2 * ( kEnd - dv ) + pt ] = c;
        }
    }
    else
    {
        // ================= helper waves =================
        const int role = wave - NP; // 0: packages (and left rows with two helpers), 1: window rows, 2: left rows
        // share of the window rows and P in H_m, coefficients as after projection m - 2 (buffer cw)
        auto windowShare = [ & ]( int m, int cw ) {
            const float* pk = sPk + ( m % BUFS ) * PKCAP;
            const float2* cs = reinterpret_cast<const float2*>( sCw + cw * 2 * VS );
            float ea = 0.f, eb = 0.f;
#pragma unroll
            for ( int i = 0; i < ( 4 * TP + 63 ) / 64; i++ )
            {
                const int t = i * 64 + lane;
                if ( t < Wc )
                {
                    const float* g = pk + ( t / TP ) * PART + t % TP;
                    const float2 cc = cs[ t ];
                    const float A = g[ 0 ];
                    ea += cc.x * A + cc.y * g[ TPQ ];
                    eb += cc.x * g[ 2 * TPQ ] + cc.y * A;
                }
            }
            const float va = waveSum( ea ), vb = waveSum( eb );
            if ( lane < 2 )
                sH[ ( m & 1 ) * 4 + lane ] = ( lane == 0 ? va : vb ) + sP[ 2 * m + lane ];
        };
        // share of the active rows that have left the window by step m - 1
        auto leftShare = [ & ]( int m ) {
            const int older = winOlder( m, newRel0, Wc ), o4 = ( older + 3 ) & ~3;
            const float* pk = sPk + ( m % BUFS ) * PKCAP + IMG + 4;
            float ea = 0.f, eb = 0.f;
#pragma unroll
            for ( int i = 0; i < kActMax / 256; i++ )
            {
                const int j = i * 256 + 4 * lane;
                if ( j < older )
                {
                    const float4 A = *reinterpret_cast<const float4*>( pk + j ), Bv = *reinterpret_cast<const float4*>( pk + o4 + j ),
                                 Cv = *reinterpret_cast<const float4*>( pk + 2 * o4 + j );
                    const float4 c0 = *reinterpret_cast<const float4*>( sC + 2 * j ), c1 = *reinterpret_cast<const float4*>( sC + 2 * j + 4 );
                    ea += c0.x * A.x + c0.y * Bv.x + c0.z * A.y + c0.w * Bv.y;
                    eb += c0.x * Cv.x + c0.y * A.x + c0.z * Cv.y + c0.w * A.y;
                    ea += c1.x * A.z + c1.y * Bv.z + c1.z * A.w + c1.w * Bv.w;
                    eb += c1.x * Cv.z + c1.y * A.z + c1.z * Cv.w + c1.w * A.w;
                }
            }
            const float va = waveSum( ea ), vb = waveSum( eb );
            if ( lane < 2 )
                sH[ ( m & 1 ) * 4 + 2 + lane ] = lane == 0 ? va : vb;
        };
        if ( role == 0 )
            waitVm<0>();
        __syncthreads();
        for ( int m = 0; m < 2 && m < K; m++ )
        {
            if ( role == 1 )
                windowShare( m, 1 );
            if ( role == NH - 1 && ( NH == 3 || role != 1 ) )
                leftShare( m );
            if ( NH == 2 && role == 0 )
                leftShare( m );
        }
        __syncthreads();
#pragma unroll 1
        for ( int k = 0; k < K; k++ )
        {
            ldsBarrier();
            // interval k: package k + BUFS goes into the buffer that step k released; H_{k+2}
            if ( role == 0 && k + BUFS < K )
                pkIssue( k + BUFS );
            if ( k + 2 < K )
            {
                if ( role == 1 )
                    windowShare( k + 2, k & 1 );
                if ( role == ( NH == 3 ? 2 : 0 ) )
                    leftShare( k + 2 );
            }
            // package k + 3 is first read after the next barrier; the younger ones stay in flight
            if ( role == 0 && k + 3 < K )
            {
                int young = 0;
#pragma unroll
                for ( int m = 4; m <= BUFS; m++ )
                    if ( k + m < K )
                        young += pkCopies( k + m );
                waitVmUpTo31( young );
            }
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
        float acc = thF[ u * L + tid ];
        for ( int ch = 0; ch < chunks; ch++ )
            acc += red[ ch * L + tid ];
        thF[ u * L + tid ] = acc;
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
