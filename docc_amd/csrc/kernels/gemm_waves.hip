// Layers, see gemm_waves.h.
#include "gemm_waves.h"

#define DOCC_GEMM_WAVES(NAME, T, BM, BN, NW, SEG, SUMS, PER_CU)                                                                                                \
    extern "C" __global__ __launch_bounds__(64 * NW, NW * PER_CU / 4) void NAME(const T* A, long lda, const T* B, long ldb, long m, long n, long k, float alpha, \
                                                                                docc_k::GemmFinish f) {                                                       \
        docc_k::gemm_waves<T, BM / 16, BN / 16, NW, SEG, 2, SUMS, 0, 0, true>(A, lda, B, ldb, m, n, k, docc_k::WavesFinish{f, alpha}, docc_k::RowsNorm{});     \
    }
DOCC_GEMM_WAVES(docc_bgemm_waves_16x16_f, uint16_t, 16, 16, 8, 8, 4, 2)
DOCC_GEMM_WAVES(docc_sgemm_waves_16x16_f, float, 16, 16, 8, 8, 16, 2)
DOCC_GEMM_WAVES(docc_bgemm_waves_32x32_f, uint16_t, 32, 32, 4, 8, 4, 2)
DOCC_GEMM_WAVES(docc_sgemm_waves_32x32_f, float, 32, 32, 4, 8, 4, 2)
DOCC_GEMM_WAVES(docc_bgemm_waves_64x64_f, uint16_t, 64, 64, 4, 4, 1, 2)
DOCC_GEMM_WAVES(docc_sgemm_waves_64x64_f, float, 64, 64, 4, 4, 2, 2)
// a work-group a compute unit: twice the ring (1024 x 1024 x 4096 in bf16 16.0 us for 19.1), twice the wavefronts (the same in fp32 67 us for 73)
DOCC_GEMM_WAVES(docc_bgemm_waves_64x64_one_f, uint16_t, 64, 64, 4, 8, 2, 1)
DOCC_GEMM_WAVES(docc_sgemm_waves_64x64_one_f, float, 64, 64, 8, 4, 2, 1)

// with the layer norm in front of up to R rows of up to 64 L vectors
#define DOCC_GEMM_WAVES_NORM(P, T, R, L, PER_CU)                                                                                                              \
    extern "C" __global__ __launch_bounds__(512, 2 * PER_CU) void docc_##P##gemm_waves_norm##L##_m##R##_f(const T* X, long ldx, const T* B, long ldb, long m,   \
                                                                                          long n, long k, float alpha, docc_k::GemmFinish f,                  \
                                                                                          docc_k::RowsNorm norm) {                                            \
        docc_k::gemm_waves<T, 1, 1, 8, 8, 2, sizeof(T) == 4 ? 16 : 4, L, R, true>(X, ldx, B, ldb, m, n, k, docc_k::WavesFinish{f, alpha}, norm);                                    \
    }
DOCC_GEMM_WAVES_NORM(b, uint16_t, 8, 4, 2)
DOCC_GEMM_WAVES_NORM(b, uint16_t, 8, 8, 1)
DOCC_GEMM_WAVES_NORM(b, uint16_t, 16, 4, 1)
DOCC_GEMM_WAVES_NORM(s, float, 8, 4, 2)
DOCC_GEMM_WAVES_NORM(s, float, 8, 8, 2)
DOCC_GEMM_WAVES_NORM(s, float, 16, 4, 2)
