// The 256 x 256 kernels on the 16x16x32 MFMA with the rest of a layer in their store (gemm_finish.h; suffix "_f").
#define DOCC_GEMM_FINISH 1
#include "gemm_async16.h"
DOCC_AGEMM16_FINISH_ONE(256, 256, 2, 2, 4, false, nn)
DOCC_AGEMM16_FINISH_ONE(256, 256, 2, 2, 4, true, nt)
