// C = act(alpha A op(B) + beta C + bias), see gemm_waves.h. fp32 1024 x 256 x 1024 12.8 us in parts on the tiles, 8.6 here;
// 8 x 8192 x 512 11.2 and 5.6; fp64 512 x 512 x 512 12.0 and 8.6.
#include "gemm_waves.h"

#define DOCC_GEMM_WAVES(P, T, S, TILE, BM, BN, NW, SEG, SUMS, PER_CU, TAG, TB)                                                                                \
    extern "C" __global__ __launch_bounds__(64 * NW, NW * PER_CU / 4) void docc_##P##gemm_waves_##TILE##_##TAG(const T* A, long lda, const T* B, long ldb, long m, long n, \
                                                                                                             long k, S alpha, S beta, S* C, long ldc, const S* bias, int act) { \
        docc_k::gemm_waves<T, BM / 16, BN / 16, NW, SEG, 2, SUMS, 0, 0, TB>(A, lda, B, ldb, m, n, k, docc_k::WavesPlain<S>{C, ldc, alpha, beta, bias, act}, docc_k::RowsNorm{}); \
    }
#define DOCC_GEMM_WAVES_BOTH(...) DOCC_GEMM_WAVES(__VA_ARGS__, nt, true) DOCC_GEMM_WAVES(__VA_ARGS__, nn, false)
DOCC_GEMM_WAVES_BOTH(s, float, float, 16x16, 16, 16, 8, 8, 16, 2)
DOCC_GEMM_WAVES_BOTH(s, float, float, 32x32, 32, 32, 4, 8, 4, 2)
DOCC_GEMM_WAVES_BOTH(s, float, float, 64x64, 64, 64, 4, 4, 2, 2)
DOCC_GEMM_WAVES_BOTH(s, float, float, 64x64_one, 64, 64, 8, 4, 2, 1)
DOCC_GEMM_WAVES_BOTH(d, double, double, 16x16, 16, 16, 8, 8, 2, 2)
DOCC_GEMM_WAVES_BOTH(d, double, double, 32x32, 32, 32, 4, 8, 2, 2)
