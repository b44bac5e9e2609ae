// bf16 x bf16 -> fp32 GEMM, asynchronous multi-stage pipeline (see gemm_async.h), tiles whose
// accumulators fit in ordinary VGPRs.
#include "gemm_async.h"

// Two tiles of 128 x 128: with stages of 64 k a work-group owns a CU (128 KB of LDS) and has 96 KB of copies in flight; with
// stages of 32 k two work-groups share it. The first is the faster one where each CU has one of them (2048^3 24.0 us against 25.4) and K
// is long (4096 x 2048 x 8192 139 against 165), the second where there are a few more tiles than CUs (1509 x 2816 x 1032 28 against 22);
// the estimate in csrc/rt/ops_gemm.cpp weighs them.
DOCC_AGEMM_CONFIG(bgemm, uint16_t, float, 128, 128, 64, 2, 2, 4)
DOCC_AGEMM_CONFIG(bgemm, uint16_t, float, 128, 128, 32, 2, 2, 4)
// Between them and the 256 x 256 tile, for products whose 256 x 256 tiles would leave CUs without one: 144 KB of LDS.
// 4096 x 2048 x 8192 (256 of these tiles) 121 us; 128 x 128 tiles 139, 256 x 256 tiles with K in two parts 139.
DOCC_AGEMM_CONFIG(bgemm, uint16_t, float, 128, 256, 64, 2, 2, 3)
#ifndef DOCC_GEMM_EPILOGUE   // tuning alternative: no epilogue variant
DOCC_AGEMM_CONFIG(bgemm, uint16_t, float, 128, 128, 64, 2, 2, 3)
#endif
