// The division of a layer norm, for the kernels that have one.
#pragma once

#include "common.h"

namespace docc_k {

// a / root, rounded once, without the ten instructions of a division for every element (bf16 4096 x 2048 with them 10.7 us, with a plain product by
// 1 / root, one rounding more, 8.3; so 8.8): q = a (1 / root) is off by a bit at most, its remainder is exact in a fused multiply-add, and what
// that adds to q rounds to the quotient (Markstein, 1990). Where the root is far from 1 (an infinity, a NaN or an underflow on the way would not
// be the quotient's) the caller divides beforehand (`direct`) and the value passes through.
struct LnQuotient {
    float root, inv;
    bool direct;
    __device__ __forceinline__ explicit LnQuotient(float r) : root(r), inv(1.0f / r), direct(!(r > 0x1p-60f && r < 0x1p60f)) {}
    __device__ __forceinline__ float operator()(float a) const {
        const float q = a * inv;
        return direct ? a : __builtin_fmaf(__builtin_fmaf(-q, root, a), inv, q);
    }
};

} // namespace docc_k
