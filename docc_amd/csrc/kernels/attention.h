// What the attention kernels share: operand types, the swizzles of the K and V blocks in LDS and the exchange between the
// two halves of a wavefront.
#pragma once

#include "gemm_mfma.h"
#include <type_traits>

namespace docc_k {

typedef uint16_t u16x8_t __attribute__((ext_vector_type(8)));
typedef uint16_t u16x4_t __attribute__((ext_vector_type(4)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef short s16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* attn_lds_ptr_t;
typedef const __attribute__((address_space(1))) void* attn_global_ptr_t;

template <>
struct Mfma<uint16_t> {
    static constexpr int VEC = 8;
    typedef u16x8_t vec_t;
};

// granule (8 bf16) index inside a row of HD / 8 granules, swizzled so that the reads below are conflict-free:
// K: sixteen lanes of a 128-bit read touch 16 consecutive rows at one granule column; V: half a wavefront of a
// transposed 64-bit read touches 4 consecutive rows x 4 granule columns. The LDS moves 256 bytes a cycle, which is
// four rows at head dim 32, two at 64 and one at 128: the swizzle spreads the rows that would meet in the same banks.
template <int HD> __device__ __forceinline__ int attn_k_swz(int row);
template <> __device__ __forceinline__ int attn_k_swz<32>(int row) { return (row >> 2) & 3; }
template <> __device__ __forceinline__ int attn_k_swz<64>(int row) { return (row >> 1) & 7; }
template <> __device__ __forceinline__ int attn_k_swz<128>(int row) { return row & 15; }
template <int HD> __device__ __forceinline__ int attn_v_swz(int row);
template <> __device__ __forceinline__ int attn_v_swz<32>(int) { return 0; }
template <> __device__ __forceinline__ int attn_v_swz<64>(int row) { return ((row >> 1) & 1) << 2; }
template <> __device__ __forceinline__ int attn_v_swz<128>(int row) { return (row & 3) << 2; }
template <int HD> __device__ __forceinline__ int attn_k_off(int row, int cv) { return (row * (HD / 8) + (cv ^ attn_k_swz<HD>(row))) * 8; }
template <int HD> __device__ __forceinline__ int attn_v_off(int row, int cv) { return (row * (HD / 8) + (cv ^ attn_v_swz<HD>(row))) * 8; }

// x of lanes 0..31 (which = 0) or of lanes 32..63 (which = 1), seen from both halves of the wave:
// v_permlane32_swap exchanges the upper half of its first operand with the lower half of its second.
// The second operand goes through an empty asm so that the compiler cannot treat the two results
// of a swap of equal inputs as equal.
__device__ __forceinline__ float half_swap(float x, int which) {
    unsigned a = __builtin_bit_cast(unsigned, x), b = a;
    asm volatile("" : "+v"(b));
    const auto sw = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    return __builtin_bit_cast(float, which ? sw[1] : sw[0]);
}

} // namespace docc_k
