// Layer normalisation over the last axis for gfx950: Y = (X - mean) / sqrt(mean((X - mean)^2) + eps) * weight + bias, fp32 or
// bf16 rows, fp32 statistics in two steps (the variance from the centred values, as the chain of nodes it stands for computes
// it). Bound by HBM: X is read once and Y written once, the row stays in registers between the two sums. As separate launches
// (cast, mean, centre and square, mean, scale) the same work moved X seven times over: [4096, 2048] bf16 in 64 us, five
// launches, against 10.9 us here. Rows of at most 32 vectors belong to that many lanes of a wavefront (a wavefront each took 226 us
// for 2^20 rows of 8 fp32, where the nodes took 62; the lanes 12.4), rows of a few KB to a wavefront (four rows a work-group, no barrier);
// longer ones, and rows too few to fill the device that way, to a work-group of 256; rows that do not fit its registers are read three times
// from L2, by one work-group a row or, from 16384 columns on, in slices.
#include "layernorm.h"

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

// sum over the TPR lanes that share a row (a power of two of neighbours); `slot`: TPR / 64 floats of LDS nobody else writes meanwhile
template <int TPR>
__device__ __forceinline__ float ln_row_sum(float v, float* slot) {
    if constexpr (TPR < 64) {
#pragma unroll
        for (int lanes = TPR / 2; lanes > 0; lanes /= 2) v += __shfl_xor(v, lanes);
        return v;
    }
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
    __shared__ float slots[2][TPR > 64 ? TPR / 64 : 1];
    const int t = threadIdx.x % TPR;
    const long row = (long) blockIdx.x * (256 / TPR) + threadIdx.x / TPR;
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
    const LnQuotient quotient(root);
    if (quotient.direct) {
#pragma unroll
        for (int i = 0; i < NV; i++)
#pragma unroll
            for (int e = 0; e < V; e++) v[i][e] /= root;
    }
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const long c = (long) (i * TPR + t) * V;
        if (c >= cols) continue;
        float w[V], b[V];
        if (W) load(reinterpret_cast<const raw*>(W), c, w);
        if (B) load(reinterpret_cast<const raw*>(B), c, b);
#pragma unroll
        for (int e = 0; e < V; e++) {
            float r = quotient(v[i][e]);
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

// Long rows, cut into gridDim.x slices of `chunk` elements (at most 256, whole vectors): a launch for the sums, one for the squares of the
// centred values, one for the result. A work-group of the latter two adds the row's parts itself, a thread a part. One
// work-group a row and the slices, fp32: a row of 2^20 1241 / 11 us, 64 rows of 64 x 56 x 56 253 / 36.
template <typename T, int V, typename F>
__device__ __forceinline__ void layernorm_slice(const void* X, long cols, long chunk, F f) {
    typedef LnElement<T> E;
    typedef typename E::raw raw;
    const raw* x = reinterpret_cast<const raw*>(X) + (long) blockIdx.y * cols;
    const long first = blockIdx.x * chunk, end = first + chunk < cols ? first + chunk : cols;
    for (long c = first + threadIdx.x * V; c < end; c += 256 * V) {
        float v[V];
        if constexpr (V == 1) {
            v[0] = E::up(x[c]);
        } else {
            const typename E::vec h = *reinterpret_cast<const typename E::vec*>(x + c);
#pragma unroll
            for (int e = 0; e < V; e++) v[e] = E::up(h[e]);
        }
        f(c, v);
    }
}

// the sum of this row's parts, in every thread
__device__ __forceinline__ float ln_parts_sum(const float* parts, float* slot) {
    return ln_row_sum<256>(threadIdx.x < gridDim.x ? parts[(long) blockIdx.y * gridDim.x + threadIdx.x] : 0.0f, slot);
}

template <typename T, int V>
__device__ __forceinline__ void layernorm_slice_sum(long cols, long chunk, const void* X, float* sums) {
    __shared__ float slots[4];
    float sum = 0.0f;
    layernorm_slice<T, V>(X, cols, chunk, [&](long, float (&v)[V]) {
#pragma unroll
        for (int e = 0; e < V; e++) sum += v[e];
    });
    sum = ln_row_sum<256>(sum, slots);
    if (threadIdx.x == 0) sums[(long) blockIdx.y * gridDim.x + blockIdx.x] = sum;
}

template <typename T, int V>
__device__ __forceinline__ void layernorm_slice_squares(long cols, long chunk, const void* X, const float* sums, float* squares) {
    __shared__ float slots[2][4];
    const float mean = ln_parts_sum(sums, slots[0]) / (float) cols;
    float sq = 0.0f;
    layernorm_slice<T, V>(X, cols, chunk, [&](long, float (&v)[V]) {
#pragma unroll
        for (int e = 0; e < V; e++) {
            const float d = v[e] - mean;
            sq += d * d;
        }
    });
    sq = ln_row_sum<256>(sq, slots[1]);
    if (threadIdx.x == 0) squares[(long) blockIdx.y * gridDim.x + blockIdx.x] = sq;
}

template <typename T, int V>
__device__ __forceinline__ void layernorm_slice_apply(long cols, long chunk, float eps, const void* X, const float* sums, const float* squares, const void* W,
                                                      const void* B, void* Y) {
    typedef LnElement<T> E;
    typedef typename E::raw raw;
    __shared__ float slots[2][4];
    const float mean = ln_parts_sum(sums, slots[0]) / (float) cols;
    const float root = sqrtf(ln_parts_sum(squares, slots[1]) / (float) cols + eps);
    raw* y = reinterpret_cast<raw*>(Y) + (long) blockIdx.y * cols;
    const raw *w = reinterpret_cast<const raw*>(W), *b = reinterpret_cast<const raw*>(B);
    const LnQuotient quotient(root);
    layernorm_slice<T, V>(X, cols, chunk, [&](long c, float (&v)[V]) {
        typename E::vec hw = {}, hb = {}, h;
        if constexpr (V > 1) {
            if (w) hw = *reinterpret_cast<const typename E::vec*>(w + c);
            if (b) hb = *reinterpret_cast<const typename E::vec*>(b + c);
        } else {
            if (w) hw[0] = w[c];
            if (b) hb[0] = b[c];
        }
#pragma unroll
        for (int e = 0; e < V; e++) {
            const float d = v[e] - mean;
            float r = quotient.direct ? d / root : quotient(d);
            if (w) r *= E::up(hw[e]);
            if (b) r += E::up(hb[e]);
            h[e] = E::down(r);
        }
        if constexpr (V > 1) *reinterpret_cast<typename E::vec*>(y + c) = h;
        else y[c] = h[0];
    });
}

} // namespace docc_k

#define DOCC_LN_ARGS long rows, long cols, float eps, const void *X, const void *W, const void *B, void *Y
// docc_layernorm_<type>_<v|s>_<w|b><NV>: vectors or single elements, a wavefront or a work-group a row; _p<lanes>: that many lanes a row, with one
// vector or four elements each
#define DOCC_LN(TYPE, T, VTAG, V, RTAG, TPR, NV)                                                                             \
    extern "C" __global__ __launch_bounds__(256) void docc_layernorm_##TYPE##_##VTAG##_##RTAG##NV(DOCC_LN_ARGS) {             \
        docc_k::layernorm_row<T, V, NV, TPR>(rows, cols, eps, X, W, B, Y);                                                   \
    }
// docc_layernorm_<type>_<v|s>_slice_<sum|squares|apply>
#define DOCC_LN_SLICE(TYPE, T, VTAG, V)                                                                                       \
    extern "C" __global__ __launch_bounds__(256) void docc_layernorm_##TYPE##_##VTAG##_slice_sum(long cols, long chunk, const void* X, float* sums) {   \
        docc_k::layernorm_slice_sum<T, V>(cols, chunk, X, sums);                                                              \
    }                                                                                                                         \
    extern "C" __global__ __launch_bounds__(256) void docc_layernorm_##TYPE##_##VTAG##_slice_squares(long cols, long chunk, const void* X,              \
                                                                                                     const float* sums, float* squares) {               \
        docc_k::layernorm_slice_squares<T, V>(cols, chunk, X, sums, squares);                                                 \
    }                                                                                                                         \
    extern "C" __global__ __launch_bounds__(256) void docc_layernorm_##TYPE##_##VTAG##_slice_apply(                           \
        long cols, long chunk, float eps, const void* X, const float* sums, const float* squares, const void* W, const void* B, void* Y) {              \
        docc_k::layernorm_slice_apply<T, V>(cols, chunk, eps, X, sums, squares, W, B, Y);                                     \
    }
#define DOCC_LN_SHORT(TYPE, T, VTAG, V, NV, TPR)                                                                             \
    extern "C" __global__ __launch_bounds__(256) void docc_layernorm_##TYPE##_##VTAG##_p##TPR(DOCC_LN_ARGS) {                 \
        docc_k::layernorm_row<T, V, NV, TPR>(rows, cols, eps, X, W, B, Y);                                                   \
    }
#define DOCC_LN_SHORTS(TYPE, T, VTAG, V, NV)  \
    DOCC_LN_SHORT(TYPE, T, VTAG, V, NV, 1)    \
    DOCC_LN_SHORT(TYPE, T, VTAG, V, NV, 2)    \
    DOCC_LN_SHORT(TYPE, T, VTAG, V, NV, 4)    \
    DOCC_LN_SHORT(TYPE, T, VTAG, V, NV, 8)    \
    DOCC_LN_SHORT(TYPE, T, VTAG, V, NV, 16)   \
    DOCC_LN_SHORT(TYPE, T, VTAG, V, NV, 32)
#define DOCC_LN_TYPE(TYPE, T, V)           \
    DOCC_LN_SHORTS(TYPE, T, v, V, 1)         \
    DOCC_LN_SHORTS(TYPE, T, s, 1, 4)         \
    DOCC_LN_SLICE(TYPE, T, v, V)             \
    DOCC_LN_SLICE(TYPE, T, s, 1)             \
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
