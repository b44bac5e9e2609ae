// The asynchronous fp32 kernels the launcher picks from (gemm_f32.hip) with the rest of a layer in their store
// (gemm_finish.h; suffix "_f").
#define DOCC_GEMM_FINISH 1
#include "gemm_async.h"
DOCC_AGEMM_FINISH_CONFIG(sgemm, float, float, 64, 64, 16, 2, 2, 4)
DOCC_AGEMM_FINISH_CONFIG(sgemm, float, float, 128, 128, 32, 2, 2, 3)
DOCC_AGEMM_FINISH_CONFIG(sgemm, float, float, 128, 256, 32, 2, 2, 2)
