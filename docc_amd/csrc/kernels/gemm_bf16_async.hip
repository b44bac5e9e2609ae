// bf16 x bf16 -> fp32 GEMM, asynchronous multi-stage pipeline (see gemm_async.h), tiles whose
// accumulators fit in ordinary VGPRs.
#include "gemm_async.h"

// Two tiles of 128 x 128: with stages of 64 k a work-group owns a CU (128 KB of LDS) and has 96 KB of copies in flight; with
// stages of 32 k two work-groups share it. Where K gives the pipeline of the first time to fill it is the faster one whether the tiles
// are one round over the CUs or several (2048^3 21.5 us against 23.0, 4096 x 2048 x 8192 139 against 165), below K = 1024 the second.
DOCC_AGEMM_CONFIG(bgemm, uint16_t, float, 128, 128, 64, 2, 2, 4)
DOCC_AGEMM_CONFIG(bgemm, uint16_t, float, 128, 128, 32, 2, 2, 4)
// Between them and the 256 x 256 tile, for products whose 256 x 256 tiles would leave CUs without one: 144 KB of LDS.
// 4096 x 2048 x 8192 (256 of these tiles) 121 us; 128 x 128 tiles 139, 256 x 256 tiles with K in two parts 139.
DOCC_AGEMM_CONFIG(bgemm, uint16_t, float, 128, 256, 64, 2, 2, 3)
#ifndef DOCC_GEMM_EPILOGUE   // tuning alternative: no epilogue variant
DOCC_AGEMM_CONFIG(bgemm, uint16_t, float, 128, 128, 64, 2, 2, 3)
#endif
