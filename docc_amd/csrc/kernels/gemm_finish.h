// The rest of a layer behind a product, applied where the product is stored:
//   out = round(act(round(alpha * A B + bias[column])) [+ residual])       fp32 arithmetic, out fp32 or bf16
// Without it the fp32 product goes to memory and a second kernel reads it back: for bf16 activations 4 + 4 + 2 bytes an
// element where 2 are needed (4096 x 8192 with bias and GELU behind K = 2048: 142 us for the product and 46 us for the pass
// behind it). The accumulators of an MFMA tile lie one column a lane, so a store straight from them would write 2-byte
// words; a wave therefore turns 64 rows of its tile at a time through its own part of LDS (free once the K loop is over) and
// works on eight consecutive columns a lane from there: bias and residual come in and the result goes out in 16-byte vectors.
#pragma once

#include "elementwise_ops.h"

namespace docc_k {

// kept in step with LinearFinish in csrc/rt/ops_gemm.cpp
struct GemmFinish {
    const void* bias;      // one value per column, or null
    const void* residual;  // dense [M][N], or null
    void* out;             // dense [M][N]
    int flags;
    int act;               // an UnaryOp (abs, relu, sigmoid, tanh), one of FinishAct, or -1
};
enum FinishFlag : int { kBiasBf16 = 1, kResidualBf16 = 2, kOutBf16 = 4, kRoundBeforeAct = 8, kRoundAfterAct = 16 };
enum FinishAct : int { kGelu = 16, kGeluTanh = 17, kSilu = 18 };

// x * Phi(x), Phi the normal distribution function: Phi(-|x|) = 2^(p(|x|) - 1) with p(a) = log2(erfc(a / sqrt 2)), here a
// polynomial of degree ten without constant term, fitted to p on [0, 5.6] by least squares reweighted towards an even error
// of 2^p; beyond it falls below p and on to -inf. One exp2 and no division. Against the fp64 value over [-9, 9]: at most 3.9e-7
// off (0.5 x (1 + erff(x / sqrt 2)) in fp32 steps: 4.5e-7), and unlike that form no cancellation for negative x.
__device__ __forceinline__ float gelu_erf(float x) {
    const float a = fabsf(x);
    float p = -3.2674233e-08f;
    p = __builtin_fmaf(p, a, 9.4363725e-07f);
    p = __builtin_fmaf(p, a, -1.1726021e-05f);
    p = __builtin_fmaf(p, a, 7.997236e-05f);
    p = __builtin_fmaf(p, a, -0.00028858453f);
    p = __builtin_fmaf(p, a, 1.1960158e-05f);
    p = __builtin_fmaf(p, a, 0.006939793f);
    p = __builtin_fmaf(p, a, -0.052440956f);
    p = __builtin_fmaf(p, a, -0.45921972f);
    p = __builtin_fmaf(p, a, -1.1511045f);
    const float tail = __builtin_amdgcn_exp2f(__builtin_fmaf(p, a, -1.0f));   // Phi(-|x|)
    return x * (x < 0.0f ? tail : 1.0f - tail);
}

// 0.5 x (1 + tanh u) = x / (1 + e^(-2u)), u = sqrt(2 / pi) (x + 0.044715 x^3)
__device__ __forceinline__ float gelu_tanh(float x) {
    const float u = 0.7978845608f * (x + 0.044715f * (x * x * x));
    return x / (1.0f + expf(-2.0f * u));
}

template <typename F>
__device__ __forceinline__ void each8(float (&v)[8], F f) {
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = f(v[e]);
}

__device__ __forceinline__ void finish_act(int act, float (&v)[8]) {
    switch (act) {   // uniform over a launch
        case kAbs: each8(v, [](float x) { return fabsf(x); }); break;
        case kReLU: each8(v, [](float x) { return fmaxf(x, 0.0f); }); break;
        case kSigmoid: each8(v, [](float x) { return 1.0f / (1.0f + expf(-x)); }); break;
        case kTanh: each8(v, [](float x) { return tanhf(x); }); break;
        case kGelu: each8(v, gelu_erf); break;
        case kGeluTanh: each8(v, gelu_tanh); break;
        case kSilu: each8(v, [](float x) { return x / (1.0f + expf(-x)); }); break;
        default: break;
    }
}

__device__ __forceinline__ float bf16_rounded(float x) { return (float) (__bf16) x; }

// eight consecutive values at `p` (bf16 or fp32), `at` in elements, 16-byte aligned
__device__ __forceinline__ void load8(const void* p, long at, bool bf16, float (&v)[8]) {
    if (bf16) {
        const bf16x8 h = *reinterpret_cast<const bf16x8*>(reinterpret_cast<const uint16_t*>(p) + at);
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = (float) h[e];
    } else {
        const f32x4* q = reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(p) + at);
        const f32x4 lo = q[0], hi = q[1];
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = lo[e], v[4 + e] = hi[e];
    }
}

// the chain on eight consecutive columns of a row; b: their bias (-0.0 where there is none), at: element index in out and residual
__device__ __forceinline__ void finish8(const GemmFinish& f, float (&v)[8], const float (&b)[8], long at) {
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] += b[e];
    if (f.flags & kRoundBeforeAct) each8(v, bf16_rounded);
    finish_act(f.act, v);
    if (f.residual) {
        if (f.flags & kRoundAfterAct) each8(v, bf16_rounded);
        float r[8];
        load8(f.residual, at, f.flags & kResidualBf16, r);
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] += r[e];
    }
    if (f.flags & kOutBf16) {
        bf16x8 h;
#pragma unroll
        for (int e = 0; e < 8; e++) h[e] = (__bf16) v[e];
        *reinterpret_cast<bf16x8*>(reinterpret_cast<uint16_t*>(f.out) + at) = h;
    } else {
        f32x4* q = reinterpret_cast<f32x4*>(reinterpret_cast<float*>(f.out) + at);
        q[0] = f32x4{v[0], v[1], v[2], v[3]};
        q[1] = f32x4{v[4], v[5], v[6], v[7]};
    }
}

// Rows of a wave tile that pass through LDS at once, and the bytes that takes per wave (rows padded by 16 bytes: the lanes of
// a wave write four or eight rows of a column block at once)
template <int TM, int TN, int MT>
struct FinishShape {
    static constexpr int IC = 64 / MT < TM ? 64 / MT : TM;
    static constexpr int LDW = TN * MT + 4;
    static constexpr int WAVE_FLOATS = IC * MT * LDW;
};

// The wave's TM x TN accumulator tiles (rows row0 .., columns col0 ..). N is a multiple of 8 and out, bias and residual are
// 16-byte aligned (the launcher sends other products through the pass of gemm_finish.hip). `buf`: FinishShape::WAVE_FLOATS
// floats of LDS of this wave alone; the caller has seen every wave's reads and copies into LDS end.
template <int TM, int TN, int MT, int NACC, typename AccT, typename RowFn>
__device__ __forceinline__ void gemm_finish_wave(const GemmFinish& f, float alpha, long M, long N, long row0, long col0, int lcol, int lane,
                                                 float* buf, AccT (&acc)[TM][TN], RowFn acc_row) {
    typedef FinishShape<TM, TN, MT> S;
    constexpr int UPR = TN * MT / 8, RPI = 64 / UPR;   // lanes across a row, rows a wave takes at once
    const int c8 = (lane % UPR) * 8, r_in = lane / UPR;
    const long col = col0 + c8;
    const bool col_ok = col < N;
    float b[8];
#pragma unroll
    for (int e = 0; e < 8; e++) b[e] = -0.0f;
    if (f.bias && col_ok) load8(f.bias, col, f.flags & kBiasBf16, b);
#pragma unroll
    for (int i0 = 0; i0 < TM; i0 += S::IC) {
#pragma unroll
        for (int i = 0; i < S::IC; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < NACC; r++) buf[(i * MT + acc_row(r)) * S::LDW + j * MT + lcol] = alpha * acc[i0 + i][j][r];
        // (a wave's LDS operations complete in order: no barrier between its own writes and reads)
        __builtin_amdgcn_wave_barrier();
#pragma unroll 2
        for (int it = 0; it < S::IC * MT / RPI; it++) {
            const int row = it * RPI + r_in;
            const f32x4* src = reinterpret_cast<const f32x4*>(buf + row * S::LDW + c8);
            const f32x4 lo = src[0], hi = src[1];
            const long grow = row0 + i0 * MT + row;
            if (grow < M && col_ok) {
                float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                finish8(f, v, b, grow * N + col);
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

} // namespace docc_k
