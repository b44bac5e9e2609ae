// A layer on a few rows: out = finish(alpha * A[m <= 16, k] B[n][k]^T), the chain of gemm_finish.h behind the product in the same launch. It reads B once
// (2 n k bytes in bf16) and is bound by that, and by what a launch costs: 8 rows x 2048 -> 8192 is 5.3 us of memory; cut along K between work-groups
// (docc_bgemm_skinny) it took 9 us and the pass that adds the parts 3 to 4.
//
// K is cut inside the work-group instead, which has 8 NT columns: eight wavefronts take pairs of lines of 128 bytes of the columns' rows in turn (single ones: 4 x 3072 -> 12288 and back in fp32 76 us for 72), loads that are an
// MFMA's operand as they come (eight consecutive k of a row in bf16, four in fp32), DEPTH lines on their way per wavefront. The 16 rows and columns of
// an MFMA are eight rows of A or B and the two halves of a line each, so that eight lanes read a whole line of a row; of the four quarters of its result
// the two where the halves meet are the product. (With 16 rows and columns and half a line of each in a load, 8 x 2048 -> 8192 took 13.0 us; it takes 9.2.) The
// wavefronts' sums meet in LDS, where a lane then finishes eight consecutive columns of a row. MT blocks of eight rows of A share the loads of B.
#include "gemm_finish.h"
#include "layernorm.h"
#include <type_traits>

namespace docc_k {

// The layer norm in front of a layer: A = (X - mean) / sqrt(mean((X - mean)^2) + eps) * weight + bias, X dense
struct RowsNorm {
    const void *weight, *bias;   // or null
    float eps;
};

// NORM > 0: rows of at most 64 NORM vectors are normalised on their way in. Every work-group does that for all of them, a wavefront a row (MT of them),
// while its first lines of B travel, and keeps the result, rounded to T as the layer norm's own store rounds it, in LDS. A launch less (3 to 4 us) for a few hundred
// instructions a wavefront: a block of 8 x 1024 19.1 us -> 17.0, of 8 x 2048 24.6 -> 23.0.
// SUMS: sets of accumulators, one line after the other to the next of them: chains of k / (16 SUMS) roundings
template <typename T, int MT, int NT, int DEPTH, int SUMS, int NORM>
__device__ __forceinline__ void gemm_rows(const T* __restrict__ A, long lda, const T* __restrict__ B, long ldb, long m, long n, long k, float alpha, const GemmFinish& f,
                                          const RowsNorm& norm) {
    constexpr bool F32 = sizeof(T) == 4;
    constexpr int NW = 8, VK = 16 / (int) sizeof(T), LINE = 8 * VK, BLOCK = 256;     // wavefronts; k of a load, k of a line; floats of a block of sums
    typedef std::conditional_t<F32, f32x4, bf16x8> vec;
    __shared__ __attribute__((aligned(16))) float sums[NW * MT * NT * BLOCK];
    __shared__ __attribute__((aligned(16))) float row[MT * 16][NT * 8 + 4];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int idx = lane & 7, k0 = ((lane >> 3 & 1) * 4 + (lane >> 4)) * VK;         // row of the operand's block, k within a line
    const long n0 = (long) blockIdx.x * (8 * NT);
    const int lines = (int) ((k + LINE - 1) / LINE);

    constexpr int kNone = (int) 0x80000000;     // beyond the end of a buffer: the load gives 0
    const long rows_left = n - n0 < 8 * NT ? n - n0 : 8 * NT;
    const auto abuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(A), 0, (int) (((m - 1) * lda + k) * (long) sizeof(T)), 0x00020000);
    const auto bbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(B) + n0 * ldb, 0, (int) (((rows_left - 1) * ldb + k) * (long) sizeof(T)), 0x00020000);
    int aoff[MT], boff[NT];
#pragma unroll
    for (int i = 0; i < MT; i++) aoff[i] = i * 8 + idx < m ? (int) ((i * 8 + idx) * lda + k0) * (int) sizeof(T) : kNone;
#pragma unroll
    for (int j = 0; j < NT; j++) boff[j] = j * 8 + idx < rows_left ? (int) ((j * 8 + idx) * ldb + k0) * (int) sizeof(T) : kNone;

    // the u-th line of this wavefront from `base` on: pairs of neighbours
    auto mine = [&](int base, int u) { return base + (u >> 1) * (2 * NW) + 2 * wave + (u & 1); };
    vec av[NORM ? 1 : DEPTH][MT], bv[DEPTH][NT];
    auto load = [&](int line, int to) {
        const bool in = line * LINE + k0 < (int) k;      // (both operands: 0 times what lies behind a row may be a NaN)
#pragma unroll
        for (int j = 0; j < NT; j++) bv[to][j] = __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b128(bbuf, in ? boff[j] : kNone, line * 128, 0));
        if constexpr (NORM == 0) {
#pragma unroll
            for (int i = 0; i < MT; i++) av[to][i] = __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b128(abuf, in ? aoff[i] : kNone, line * 128, 0));
        }
    };
    // NORM: the normalised rows, a vector further apart than they are long (eight lanes read eight rows)
    extern __shared__ __attribute__((aligned(16))) unsigned char rows_lds[];
    T* const normed = reinterpret_cast<T*>(rows_lds);
    const int pitch = (int) k + VK;
    auto from_lds = [&](int line, int i) {
        const bool in = line * LINE + k0 < (int) k;
        const vec v = *reinterpret_cast<const vec*>(normed + (i * 8 + idx) * pitch + (in ? line * LINE + k0 : 0));
        return in ? v : vec{};
    };
    static_assert(DEPTH % SUMS == 0, "a line's set of accumulators is known at compile time");
    f32x4 acc[SUMS][MT][NT];
#pragma unroll
    for (int u = 0; u < SUMS; u++)
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++) acc[u][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (NORM > 0) {
        // the rows and the norm's operands first: loads arrive in the order they were issued in
        vec x[MT][NORM], w[NORM], b[NORM];
        const int last_vector = (int) k / VK;
        auto at = [&](int i) { return i * 64 + lane < last_vector ? (i * 64 + lane) * VK : 0; };
#pragma unroll
        for (int r = 0; r < MT; r++)
#pragma unroll
            for (int i = 0; i < NORM; i++) x[r][i] = *reinterpret_cast<const vec*>(A + (r * 8 + wave < m ? r * 8 + wave : 0) * lda + at(i));
#pragma unroll
        for (int i = 0; i < NORM; i++) {
            if (norm.weight) w[i] = *reinterpret_cast<const vec*>(reinterpret_cast<const T*>(norm.weight) + at(i));
            if (norm.bias) b[i] = *reinterpret_cast<const vec*>(reinterpret_cast<const T*>(norm.bias) + at(i));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < DEPTH; u++) load(mine(0, u), u);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < MT; r++) {
            float v[NORM][VK], sum = 0.f, sq = 0.f;
#pragma unroll
            for (int i = 0; i < NORM; i++)
#pragma unroll
                for (int e = 0; e < VK; e++) {
                    v[i][e] = i * 64 + lane < last_vector ? (float) x[r][i][e] : 0.f;
                    sum += v[i][e];
                }
            const float mean = wave_sum(sum) / (float) k;
#pragma unroll
            for (int i = 0; i < NORM; i++)
#pragma unroll
                for (int e = 0; e < VK; e++) {
                    v[i][e] -= mean;
                    if (i * 64 + lane < last_vector) sq += v[i][e] * v[i][e];
                }
            const float root = sqrtf(wave_sum(sq) / (float) k + norm.eps);
            const LnQuotient quotient(root);
#pragma unroll
            for (int i = 0; i < NORM; i++) {
                vec out;
#pragma unroll
                for (int e = 0; e < VK; e++) {
                    float y = quotient.direct ? v[i][e] / root : quotient(v[i][e]);
                    if (norm.weight) y *= (float) w[i][e];
                    if (norm.bias) y += (float) b[i][e];
                    if constexpr (F32) out[e] = y;
                    else out[e] = (__bf16) y;
                }
                if (i * 64 + lane < last_vector) *reinterpret_cast<vec*>(normed + (r * 8 + wave) * pitch + (i * 64 + lane) * VK) = r * 8 + wave < m ? out : vec{};
            }
        }
        __syncthreads();
    } else {
#pragma unroll
        for (int u = 0; u < DEPTH; u++) load(mine(0, u), u);
    }
    for (int base = 0; base < lines; base += DEPTH * NW) {
#pragma unroll
        for (int u = 0; u < DEPTH; u++) {
            constexpr bool FROM_LDS = NORM > 0;
            const int a = FROM_LDS ? 0 : u;
            if constexpr (FROM_LDS) {
#pragma unroll
                for (int i = 0; i < MT; i++) av[0][i] = from_lds(mine(base, u), i);
            }
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    if constexpr (F32) {
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[u % SUMS][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[a][i][e], bv[u][j][e], acc[u % SUMS][i][j], 0, 0, 0);
                    } else {
                        acc[u % SUMS][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[a][i], bv[u][j], acc[u % SUMS][i][j], 0, 0, 0);
                    }
                }
            if (mine(base + DEPTH * NW, u) < lines) load(mine(base + DEPTH * NW, u), u);
            else if constexpr (!FROM_LDS) {
#pragma unroll
                for (int i = 0; i < MT; i++) av[u][i] = vec{};
            }
        }
    }
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) {
#pragma unroll
            for (int u = SUMS / 2; u >= 1; u /= 2)
#pragma unroll
                for (int q = 0; q < u; q++) acc[q][i][j] += acc[q + u][i][j];
            *reinterpret_cast<f32x4*>(sums + ((wave * MT + i) * NT + j) * BLOCK + lane * 4) = acc[0][i][j];
        }
    __syncthreads();
    // Register r of lane l is row 4 (l / 16) + r, column l % 16 of a block. A thread adds up one value of a row and column and half, then the halves meet.
    static_assert(MT * NT * 128 <= 64 * NW, "a thread a value");
    if (tid < MT * NT * 128) {
        const int block = tid >> 7, q = (tid >> 3) & 15, col = tid & 7;      // q: row of the block, its half is q / 8
        const float* from = sums + block * BLOCK + ((q >> 2) * 16 + (q >> 3) * 8 + col) * 4 + (q & 3);
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < NW; w++) v += from[w * (MT * NT * BLOCK)];
        row[block / NT * 16 + q][block % NT * 8 + col] = v;
    }
    __syncthreads();
    if (tid < MT * 8 * NT) {
        const int t = tid / NT, c8 = tid % NT * 8;
        const long col = n0 + c8;
        if (t < m && col < n) {
            float v[8], b[8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                v[e] = alpha * (row[(t >> 3) * 16 + (t & 7)][c8 + e] + row[(t >> 3) * 16 + 8 + (t & 7)][c8 + e]);
                asm volatile("" : "+v"(v[e]));    // the product is rounded before the bias is added
                b[e] = -0.0f;
            }
            if (f.bias) load8(f.bias, col, f.flags & kBiasBf16, b);
            finish8(f, v, b, t * n + col);
        }
    }
}

} // namespace docc_k

#define DOCC_GEMM_ROWS(P, T, MT, NT, DEPTH, SUMS)                                                                                                              \
    extern "C" __global__ __launch_bounds__(512) void docc_##P##gemm_rows_m##MT##_n##NT##_f(const T* A, long lda, const T* B, long ldb, long m, long n, long k,  \
                                                                                           float alpha, docc_k::GemmFinish f) {                                \
        docc_k::gemm_rows<T, MT, NT, DEPTH, SUMS, 0>(A, lda, B, ldb, m, n, k, alpha, f, docc_k::RowsNorm{});                                                    \
    }
DOCC_GEMM_ROWS(b, uint16_t, 1, 1, 8, 2)
DOCC_GEMM_ROWS(b, uint16_t, 1, 2, 4, 2)
DOCC_GEMM_ROWS(b, uint16_t, 2, 1, 4, 2)
DOCC_GEMM_ROWS(b, uint16_t, 2, 2, 4, 2)
DOCC_GEMM_ROWS(b, uint16_t, 4, 1, 2, 2)
DOCC_GEMM_ROWS(s, float, 1, 1, 8, 4)
DOCC_GEMM_ROWS(s, float, 1, 2, 4, 4)
DOCC_GEMM_ROWS(s, float, 2, 1, 4, 4)
DOCC_GEMM_ROWS(s, float, 2, 2, 4, 4)
DOCC_GEMM_ROWS(s, float, 4, 1, 2, 2)

// with the layer norm in front, rows of up to 64 L vectors
#define DOCC_GEMM_ROWS_NORM(P, T, MT, NT, DEPTH, SUMS, L)                                                                                                      \
    extern "C" __global__ __launch_bounds__(512, MT == 1 && L == 4 ? 4 : 2) void docc_##P##gemm_rows_m##MT##_n##NT##_norm##L##_f(const T* X, long ldx, const T* B, long ldb, long m,        \
                                                                                                     long n, long k, float alpha, docc_k::GemmFinish f,       \
                                                                                                     docc_k::RowsNorm norm) {                                 \
        docc_k::gemm_rows<T, MT, NT, DEPTH, SUMS, L>(X, ldx, B, ldb, m, n, k, alpha, f, norm);                                                                 \
    }
DOCC_GEMM_ROWS_NORM(b, uint16_t, 1, 1, 8, 2, 4)
DOCC_GEMM_ROWS_NORM(b, uint16_t, 1, 2, 4, 2, 4)
DOCC_GEMM_ROWS_NORM(b, uint16_t, 1, 1, 8, 2, 8)
DOCC_GEMM_ROWS_NORM(b, uint16_t, 1, 2, 4, 2, 8)
DOCC_GEMM_ROWS_NORM(b, uint16_t, 2, 1, 4, 2, 4)
DOCC_GEMM_ROWS_NORM(b, uint16_t, 2, 2, 4, 2, 4)
DOCC_GEMM_ROWS_NORM(s, float, 1, 1, 8, 4, 4)
DOCC_GEMM_ROWS_NORM(s, float, 1, 2, 4, 4, 4)
DOCC_GEMM_ROWS_NORM(s, float, 1, 1, 8, 4, 8)
DOCC_GEMM_ROWS_NORM(s, float, 1, 2, 4, 4, 8)
DOCC_GEMM_ROWS_NORM(s, float, 2, 1, 4, 4, 4)
