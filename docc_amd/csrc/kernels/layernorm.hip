// Layer normalisation over the last axis for gfx950: Y = (X - mean) / sqrt(mean((X - mean)^2) + eps) * weight + bias, fp32 or
// bf16 rows, fp32 statistics in two steps (the variance from the centred values, as the chain of nodes it stands for computes
// it). Bound by HBM: X is read once and Y written once, the row stays in registers between the two sums. As separate launches
// (cast, mean, centre and square, mean, scale) the same work moved X seven times over: [4096, 2048] bf16 in 64 us, five
// launches, against 12.8 us here. Rows of a few KB belong to a wavefront (four rows a work-group, no barrier); longer ones, and rows too few to fill the
// device that way, to a work-group of 256; rows that do not fit its registers are read three times from L2.
#include "common.h"

namespace docc_k {

template <typename T> struct LnElement;
template <> struct LnElement<float> {
    typedef float raw;
    typedef f32x4 vec;
    static constexpr int VEC = 4;
    static __device__ __forceinline__ float up(float v) { return v; }
    static __device__ __forceinline__ float down(float v) { return v; }
};
template <> struct LnElement<uint16_t> {
    typedef __bf16 raw;
    typedef bf16x8 vec;
    static constexpr int VEC = 8;
    static __device__ __forceinline__ float up(__bf16 v) { return (float) v; }
    static __device__ __forceinline__ __bf16 down(float v) { return (__bf16) v; }
};

// sum over the TPR lanes that share a row; `slot`: TPR / 64 floats of LDS nobody else writes meanwhile
template <int TPR>
__device__ __forceinline__ float ln_row_sum(float v, float* slot) {
    v = wave_sum(v);
    if (TPR == 64) return v;
    if ((threadIdx.x & 63) == 0) slot[threadIdx.x >> 6] = v;
    __syncthreads();
    float s = slot[0];
#pragma unroll
    for (int w = 1; w < TPR / 64; w++) s += slot[w];
    return s;
}

// NV vectors of V elements a lane, TPR lanes a row; cols <= TPR * NV * V and a multiple of V
template <typename T, int V, int NV, int TPR>
__device__ __forceinline__ void layernorm_row(long rows, long cols, float eps, const void* X, const void* W, const void* B, void* Y) {
    typedef LnElement<T> E;
    typedef typename E::raw raw;
    __shared__ float slots[2][TPR / 64];
    const int t = threadIdx.x % TPR;
    const long row = TPR == 64 ? (long) blockIdx.x * 4 + (threadIdx.x >> 6) : (long) blockIdx.x;
    if (row >= rows) return;
    const raw* x = reinterpret_cast<const raw*>(X) + row * cols;
    raw* y = reinterpret_cast<raw*>(Y) + row * cols;
    auto load = [&](const raw* p, long c, float (&v)[V]) {
        if constexpr (V == 1) {
            v[0] = E::up(p[c]);
        } else {
            const typename E::vec h = *reinterpret_cast<const typename E::vec*>(p + c);
#pragma unroll
            for (int e = 0; e < V; e++) v[e] = E::up(h[e]);
        }
    };
    float v[NV][V];
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const long c = (long) (i * TPR + t) * V;
        if (c < cols) load(x, c, v[i]);
        else
#pragma unroll
            for (int e = 0; e < V; e++) v[i][e] = 0.0f;
#pragma unroll
        for (int e = 0; e < V; e++) sum += v[i][e];
    }
    const float mean = ln_row_sum<TPR>(sum, slots[0]) / (float) cols;
    float sq = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; i++)
        if ((long) (i * TPR + t) * V < cols) {
#pragma unroll
            for (int e = 0; e < V; e++) {
                v[i][e] -= mean;
                sq += v[i][e] * v[i][e];
            }
        }
    const float root = sqrtf(ln_row_sum<TPR>(sq, slots[1]) / (float) cols + eps);
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const long c = (long) (i * TPR + t) * V;
        if (c >= cols) continue;
        float w[V], b[V];
        if (W) load(reinterpret_cast<const raw*>(W), c, w);
        if (B) load(reinterpret_cast<const raw*>(B), c, b);
#pragma unroll
        for (int e = 0; e < V; e++) {
            float r = v[i][e] / root;
            if (W) r *= w[e];
            if (B) r += b[e];
            v[i][e] = r;
        }
        if constexpr (V == 1) {
            y[c] = E::down(v[i][0]);
        } else {
            typename E::vec h;
#pragma unroll
            for (int e = 0; e < V; e++) h[e] = E::down(v[i][e]);
            *reinterpret_cast<typename E::vec*>(y + c) = h;
        }
    }
}

// any length: a work-group of 1024 reads the row once per sum and once for the result
template <typename T>
__device__ __forceinline__ void layernorm_long(long cols, float eps, const void* X, const void* W, const void* B, void* Y) {
    typedef LnElement<T> E;
    typedef typename E::raw raw;
    __shared__ float slots[2][16];
    const raw* x = reinterpret_cast<const raw*>(X) + (long) blockIdx.x * cols;
    raw* y = reinterpret_cast<raw*>(Y) + (long) blockIdx.x * cols;
    const raw *w = reinterpret_cast<const raw*>(W), *b = reinterpret_cast<const raw*>(B);
    float sum = 0.0f;
    for (long c = threadIdx.x; c < cols; c += 1024) sum += E::up(x[c]);
    const float mean = ln_row_sum<1024>(sum, slots[0]) / (float) cols;
    float sq = 0.0f;
    for (long c = threadIdx.x; c < cols; c += 1024) {
        const float d = E::up(x[c]) - mean;
        sq += d * d;
    }
    const float root = sqrtf(ln_row_sum<1024>(sq, slots[1]) / (float) cols + eps);
    for (long c = threadIdx.x; c < cols; c += 1024) {
        float r = (E::up(x[c]) - mean) / root;
        if (w) r *= E::up(w[c]);
        if (b) r += E::up(b[c]);
        y[c] = E::down(r);
    }
}

} // namespace docc_k

#define DOCC_LN_ARGS long rows, long cols, float eps, const void *X, const void *W, const void *B, void *Y
// docc_layernorm_<type>_<v|s>_<w|b><NV>: vectors or single elements, a wavefront or a work-group a row
#define DOCC_LN(TYPE, T, VTAG, V, RTAG, TPR, NV)                                                                             \
    extern "C" __global__ __launch_bounds__(256) void docc_layernorm_##TYPE##_##VTAG##_##RTAG##NV(DOCC_LN_ARGS) {             \
        docc_k::layernorm_row<T, V, NV, TPR>(rows, cols, eps, X, W, B, Y);                                                   \
    }
#define DOCC_LN_TYPE(TYPE, T, V)           \
    DOCC_LN(TYPE, T, v, V, w, 64, 1)         \
    DOCC_LN(TYPE, T, v, V, w, 64, 2)         \
    DOCC_LN(TYPE, T, v, V, w, 64, 4)         \
    DOCC_LN(TYPE, T, v, V, b, 256, 1)        \
    DOCC_LN(TYPE, T, v, V, b, 256, 2)        \
    DOCC_LN(TYPE, T, v, V, b, 256, 4)        \
    DOCC_LN(TYPE, T, s, 1, w, 64, 4)         \
    DOCC_LN(TYPE, T, s, 1, b, 256, 4)        \
    DOCC_LN(TYPE, T, s, 1, b, 256, 16)       \
    extern "C" __global__ __launch_bounds__(1024) void docc_layernorm_##TYPE##_long(DOCC_LN_ARGS) {                           \
        docc_k::layernorm_long<T>(cols, eps, X, W, B, Y);                                                                    \
    }
DOCC_LN_TYPE(f32, float, 4)
DOCC_LN_TYPE(bf16, uint16_t, 8)
DOCC_LN(f32, float, v, 4, b, 256, 8)
