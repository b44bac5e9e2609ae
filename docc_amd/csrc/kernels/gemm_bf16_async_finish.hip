// The kernels of gemm_bf16_async.hip with the rest of a layer in their store (gemm_finish.h; suffix "_f").
#define DOCC_GEMM_FINISH 1
#include "gemm_async.h"
DOCC_AGEMM_FINISH_CONFIG(bgemm, uint16_t, float, 128, 128, 32, 2, 2, 4)
DOCC_AGEMM_FINISH_CONFIG(bgemm, uint16_t, float, 128, 128, 64, 2, 2, 4)
DOCC_AGEMM_FINISH_CONFIG(bgemm, uint16_t, float, 128, 256, 64, 2, 2, 3)
