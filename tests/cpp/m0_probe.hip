// A copy to LDS by the compiler (which keeps its LDS address in M0), one by dmaDwordx4 or dmaDword, and
// the compiler's again at the first address: the compiler has to set M0 anew after ours.
#include "apsm_train2.h"

template <int KIND>
__device__ __forceinline__ void probe( const float* a, float* out )
{
    __shared__ float lds[ 1024 ];
    typedef __attribute__( ( address_space( 1 ) ) ) const unsigned* G;
    typedef __attribute__( ( address_space( 3 ) ) ) unsigned* L;
    const uint32_t at = __builtin_amdgcn_readfirstlane( (uint32_t)(uintptr_t)( __attribute__( ( address_space( 3 ) ) ) float* )lds );
    __builtin_amdgcn_global_load_lds( (G)( a + threadIdx.x ), (L)lds, 4, 0, 0 );
    if ( KIND == 0 )
        apsm::dmaDword( a + 64 + threadIdx.x, at + 2048u );
    else
        apsm::dmaDwordx4( a + 64, 16u * threadIdx.x, at + 2048u );
    __builtin_amdgcn_global_load_lds( (G)( a + 512 + threadIdx.x ), (L)lds, 4, 0, 0 );
    __syncthreads();
    out[ threadIdx.x ] = lds[ threadIdx.x ] + lds[ 512 + threadIdx.x ];
}

extern "C" __global__ void probe_dword( const float* a, float* out ) { probe<0>( a, out ); }
extern "C" __global__ void probe_dwordx4( const float* a, float* out ) { probe<1>( a, out ); }
