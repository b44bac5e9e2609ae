// Operands and extents of a 2-d convolution; must match ConvParams and ConvFinish in csrc/rt/ops_conv.cpp.
#pragma once

namespace docc_k {

struct ConvParams {
    const float* X;
    const float* Wt;
    const float* bias;
    float* Y;
    int N, C, H, W, OC, KH, KW, OH, OW;
    int stride_h, stride_w, pad_h, pad_w, dil_h, dil_w;
    // channels of the tensors X and Y lie in: C and OC, or more when the call is one group of a grouped convolution (the
    // images are then XC and YC channels apart)
    int XC, YC;
    // grouped convolution in one launch (the entry points with the suffix _g): blockIdx.z is the group, whose operands lie
    // these many elements further on. The kernels of a single convolution do not look at them (their registers are full).
    long GX, GW, GB, GY;
};

// The rest of a layer behind a convolution, applied where it is stored: Y = act(convolution + bias + residual).
struct ConvFinish {
    const float* residual;   // dense like Y, or null
    int relu;
};
__device__ __forceinline__ float conv_finished(const ConvFinish& f, float v, float residual) {
    v += residual;           // -0.0 where there is none: no value changes
    return f.relu ? fmaxf(v, 0.0f) : v;
}

// Work-groups are dealt to the 8 XCDs in turn: number them so that an XCD gets consecutive ones (whose work shares input).
__device__ __forceinline__ int xcd_contiguous(int id, int n) {
    const int xcd = id & 7, q = n >> 3, r = n & 7;
    return xcd * q + (xcd < r ? xcd : r) + (id >> 3);
}

} // namespace docc_k
