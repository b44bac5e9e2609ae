// Operands whose rows do not start on 16-byte boundaries (or whose contiguous extent is no whole number of vectors), copied into the
// form the asynchronous GEMM kernels read: [rows][kp] with k contiguous, kp >= k a whole number of vectors, zeros behind k. Without
// it such products ran on the element-wise loaders of gemm_mfma.h / gemm_bf16.hip, bf16 4096 x 4097 x 4096 in 1146 us and 300 x 300 x
// 8001 fp32 in 415; the copy is bound by HBM (read and write once, a tenth of such a product's time or less).
// One launch packs both operands of a product: work-groups [0, groups_a) take A, the others B. A tile is 64 rows of the result by 64 k.
// A source stored [k][rows] is turned in LDS; one stored [rows][k] is copied, a lane reading the vector it writes element by
// element (the elements of a line come out of L1).
#include "common.h"

namespace docc_k {

struct PackSource {
    const void* src;
    void* dst;
    long ld, rows;
    int k_major;   // stored [k][ld] instead of [rows][ld]
};

template <typename U>
__device__ __forceinline__ void pack_tile(const PackSource& p, long tile, long k, long kp) {
    constexpr int V = 16 / (int) sizeof(U), PER_ROW = 64 / V;   // vectors across the 64 k of a tile's row
    typedef U vec_t __attribute__((ext_vector_type(V)));
    __shared__ U turned[64][64 + 1];
    const long tiles_k = (kp + 63) / 64;
    const long r0 = tile / tiles_k * 64, k0 = tile % tiles_k * 64;
    const U* src = reinterpret_cast<const U*>(p.src);
    U* dst = reinterpret_cast<U*>(p.dst);
    const int tid = threadIdx.x;
    // every load of the tile is issued before the first store: one wait for memory, not one per row
    if (p.k_major) {
        const int c = tid & 63;
        U in[16];
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const long kk = k0 + (tid >> 6) + 4 * i;
            in[i] = kk < k && r0 + c < p.rows ? src[kk * p.ld + r0 + c] : (U) 0;
        }
#pragma unroll
        for (int i = 0; i < 16; i++) turned[(tid >> 6) + 4 * i][c] = in[i];
        __syncthreads();
    }
    constexpr int UNITS = 64 * PER_ROW / 256;
    vec_t v[UNITS];
#pragma unroll
    for (int i = 0; i < UNITS; i++) {
        const int row = (tid + 256 * i) / PER_ROW, kc = (tid + 256 * i) % PER_ROW * V;
#pragma unroll
        for (int e = 0; e < V; e++)
            v[i][e] = p.k_major ? turned[kc + e][row] : r0 + row < p.rows && k0 + kc + e < k ? src[(r0 + row) * p.ld + k0 + kc + e] : (U) 0;
    }
#pragma unroll
    for (int i = 0; i < UNITS; i++) {
        const int row = (tid + 256 * i) / PER_ROW, kc = (tid + 256 * i) % PER_ROW * V;
        if (r0 + row < p.rows && k0 + kc < kp) *reinterpret_cast<vec_t*>(dst + (r0 + row) * kp + k0 + kc) = v[i];
    }
}

} // namespace docc_k

#define DOCC_GEMM_PACK(BYTES, U)                                                                                              \
    extern "C" __global__ __launch_bounds__(256) void docc_gemm_pack_b##BYTES(docc_k::PackSource a, docc_k::PackSource b,    \
                                                                              long groups_a, long k, long kp) {              \
        const long g = blockIdx.x;                                                                                            \
        docc_k::pack_tile<U>(g < groups_a ? a : b, g < groups_a ? g : g - groups_a, k, kp);                                   \
    }
DOCC_GEMM_PACK(2, uint16_t)
DOCC_GEMM_PACK(4, uint32_t)
DOCC_GEMM_PACK(8, uint64_t)
