// The FP32 detect's largest register users in a translation unit of their own.
#include "apsm_detect_mfma.h"

template __global__ void apsm::apsm_detect_mfma<32, 14, apsm::PREC_F32>( const float*, int64_t, const float*, const float*, const float*, int64_t,
                                                                         const float*, int64_t, int, float, float, float, float*, int );
template __global__ void apsm::apsm_detect_mfma<32, 16, apsm::PREC_F32>( const float*, int64_t, const float*, const float*, const float*, int64_t,
                                                                         const float*, int64_t, int, float, float, float, float*, int );
