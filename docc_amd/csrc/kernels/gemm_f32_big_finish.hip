// The 256 x 256 fp32 kernels (gemm_f32_big.hip) with the rest of a layer in their store (gemm_finish.h; suffix "_f").
#define DOCC_GEMM_FINISH 1
#include "gemm_async.h"
DOCC_AGEMM_FINISH_CONFIG(sgemm, float, float, 256, 256, 32, 2, 2, 2)
