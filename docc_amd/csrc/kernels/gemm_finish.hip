// The chain of gemm_finish.h on a product that is in memory already: the parts of a product whose K was cut (added in order,
// as docc_splitk_combine_f32 does), and products of the kernels that have no such store (matrix-vector kernels, operands off a
// 16-byte boundary). Bound by reading the fp32 parts and writing the result.
#include "gemm_finish.h"

namespace docc_k {

// P: `splits` fp32 matrices [M][N]. V = 8: whole vectors (N a multiple of 8, 16-byte aligned pointers), else one element a lane.
template <int V>
__device__ __forceinline__ void finish_parts(const float* __restrict__ P, long M, long N, int splits, float alpha, const GemmFinish& f) {
    const long total = M * N, units = total / V;
    const long stride = (long) gridDim.x * 256;
    for (long u = (long) blockIdx.x * 256 + threadIdx.x; u < units; u += stride) {
        const long at = u * V, col = at % N;
        if constexpr (V == 8) {
            float v[8];
            load8(P, at, false, v);
            for (int z = 1; z < splits; z++) {
                float w[8];
                load8(P, (long) z * total + at, false, w);
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] += w[e];
            }
            float b[8];
#pragma unroll
            for (int e = 0; e < 8; e++) b[e] = -0.0f, v[e] *= alpha;
            if (f.bias) load8(f.bias, col, f.flags & kBiasBf16, b);
            // the product is rounded before the bias is added, as in the store of the kernels
#pragma unroll
            for (int e = 0; e < 8; e++) asm volatile("" : "+v"(v[e]));
            finish8(f, v, b, at);
        } else {
            auto one = [&](const void* p, long i, bool bf16) {
                return bf16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(p)[i]) : reinterpret_cast<const float*>(p)[i];
            };
            float s = P[at];
            for (int z = 1; z < splits; z++) s += P[(long) z * total + at];
            s *= alpha;
            asm volatile("" : "+v"(s));
            if (f.bias) s += one(f.bias, col, f.flags & kBiasBf16);
            float v[8] = {s, 0, 0, 0, 0, 0, 0, 0};
            if (f.flags & kRoundBeforeAct) v[0] = bf16_rounded(v[0]);
            finish_act(f.act, v);
            if (f.residual) {
                if (f.flags & kRoundAfterAct) v[0] = bf16_rounded(v[0]);
                v[0] += one(f.residual, at, f.flags & kResidualBf16);
            }
            if (f.flags & kOutBf16) reinterpret_cast<uint16_t*>(f.out)[at] = __builtin_bit_cast(uint16_t, (__bf16) v[0]);
            else reinterpret_cast<float*>(f.out)[at] = v[0];
        }
    }
}

} // namespace docc_k

extern "C" __global__ __launch_bounds__(256) void docc_gemm_finish_v8(const float* P, long M, long N, int splits, float alpha, docc_k::GemmFinish f) {
    docc_k::finish_parts<8>(P, M, N, splits, alpha, f);
}
extern "C" __global__ __launch_bounds__(256) void docc_gemm_finish_v1(const float* P, long M, long N, int splits, float alpha, docc_k::GemmFinish f) {
    docc_k::finish_parts<1>(P, M, N, splits, alpha, f);
}
