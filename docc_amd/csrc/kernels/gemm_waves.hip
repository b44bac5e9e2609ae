// A layer on few rows, or any whose product has too few tiles to fill the compute units: out = finish(alpha * A[m, k] B[n][k]^T), the chain of gemm_finish.h behind
// the product in the same launch. On a few rows it reads B once and is bound by that (8 rows x 2048 -> 8192 in bf16: 5.3 us of memory, 7.8 measured); with a few hundred it
// is bound by its launch and by how long the first bytes take: a tile a work-group on the kernels of gemm_async.h leaves a wavefront a SIMD, which waits for every K-step's
// copies at a barrier (1024 x 256 x 1024 13.8 us in bf16, 13.1 in fp32, K in parts and a pass behind them), and cutting K between work-groups takes a second launch of
// 3 to 4 us.
//
// K is cut between the NW wavefronts of the work-group instead: each takes pieces of 16 SEG bytes of the tile's rows and columns in turn and has the whole tile's sums in
// registers. No operand is read twice in a work-group that way, and there is no barrier before the end: a wavefront copies its pieces into a ring of its own in LDS, two
// of them on their way (1024 x 256 x 1024 5.3 us, 8.6 in fp32).
// (Straight into registers, as an MFMA takes them, 16 lanes side by side read 16 rows: 15 bytes a clock and compute unit, 32 x 32 tiles of 2048 k 18.7 us in fp32 for
// 13.0. Eight wavefronts on the 32 x 32 tile, half as deep pieces and longer rings were no faster; 16 x 32 tiles like those of 16 x 16.)
// The wavefronts' sums meet in LDS, where a lane then finishes eight consecutive columns of a row.
#include "gemm_finish.h"
#include "gemm_async.h"
#include "layernorm.h"
#include <type_traits>

namespace docc_k {

// The layer norm in front of a layer: A = (X - mean) / sqrt(mean((X - mean)^2) + eps) * weight + bias, X dense
struct RowsNorm {
    const void *weight, *bias;   // or null
    float eps;
};

// Blocks of 16 rows and columns: MB x NB of them are the tile. Rows of a piece lie one behind the other in a stage of the ring, the granules of 16 bytes XORed by the row:
// eight lanes read eight rows without bank conflicts. SUMS sets of accumulators: chains of k / (NW SUMS) products.
//
// NORM > 0 (a tile of MR <= 16 rows, all there are): rows of at most 64 NORM vectors are normalised on their way in. Every work-group does that for all of them, a
// wavefront a row, while its first pieces of B travel, and keeps the result, rounded to T as the layer norm's own store rounds it, in LDS behind the rings: a launch less
// for a few hundred instructions a wavefront (a block on 8 x 2048 in bf16 24.6 us with the launch, 23.0 without, both on an earlier kernel).
template <typename T, int MB, int NB, int NW, int SEG, int STAGES, int SUMS, int NORM, int MR>
__device__ __forceinline__ void gemm_waves(const T* __restrict__ A, long lda, const T* __restrict__ B, long ldb, long m, long n, long k, float alpha, const GemmFinish& f,
                                           const RowsNorm& norm) {
    constexpr bool F32 = sizeof(T) == 4;
    constexpr int VK = 16 / (int) sizeof(T), PIECE = SEG * VK, BM = 16 * MB, BN = 16 * NB, LDW = BN + 4;
    constexpr int BC = NORM ? 0 : BM;      // rows of A that are copied
    constexpr int STAGE = (BC + BN) * SEG * 16, NL = (BC + BN) * SEG / 64, RPL = 64 / SEG;    // bytes, copies and a copy's rows of a stage
    constexpr bool TWICE = NW * BM * LDW * 4 > 65536;      // the sums of half of the wavefronts at a time
    constexpr int COPIES = TWICE ? NW / 2 : NW;
    static_assert((SEG == 4 || SEG == 8) && (STAGES - 1) * NL < 64, "the swizzles; vmcnt holds at most 63 outstanding copies");
    static_assert(SUMS == 1 || (F32 ? SUMS % 4 == 0 || SUMS == 2 : SUMS == 2 || (SUMS == 4 && SEG == 8)), "a product's set is known at compile time");
    static_assert(NORM == 0 || (MB == 1 && MR <= 16), "the rows that are normalised");
    typedef std::conditional_t<F32, f32x4, bf16x8> vec;
    extern __shared__ __attribute__((aligned(16))) unsigned char waves_lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int idx = lane & 15, grp = lane >> 4;
    int tm, tn;
    gemm_tile_coords(blockIdx.x, (int) ((m + BM - 1) / BM), (int) ((n + BN - 1) / BN), tm, tn);
    const long m0 = (long) tm * BM, n0 = (long) tn * BN;
    const int rows = m - m0 < BM ? (int) (m - m0) : BM, cols = n - n0 < BN ? (int) (n - n0) : BN;
    const int pieces = (int) ((k + PIECE - 1) / PIECE), kleft = (int) (k - (long) (pieces - 1) * PIECE);   // k of the last piece
    auto swz = [](int row) { return SEG == 8 ? row & 7 : (row >> 2) & 3; };

    // copy i of a stage: rows RPL i .. of the tile's BM + BN, those beyond the edge as copies of the last (their products are not stored)
    unsigned off[NL], off_last[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const bool is_a = i * RPL < BC;
        const int row = (is_a ? i * RPL : i * RPL - BC) + lane / SEG, granule = (lane % SEG) ^ swz(row);
        const int r = is_a ? (row < rows ? row : rows - 1) : (row < cols ? row : cols - 1);
        off[i] = (unsigned) r * (unsigned) ((is_a ? lda : ldb) * (long) sizeof(T)) + granule * 16;
        off_last[i] = off[i] - (granule * VK < kleft ? 0 : granule * 16);     // behind the end of K: the first of the row, cleared in registers
    }
    const char* const abase = reinterpret_cast<const char*>(A + m0 * lda);
    const char* const bbase = reinterpret_cast<const char*>(B + n0 * ldb);
    unsigned char* const ring = waves_lds + wave * (STAGES * STAGE);
    auto copy = [&](int piece, int stage) {
        const long at = (long) piece * (16 * SEG);
        const bool last = piece == pieces - 1;
#pragma unroll
        for (int i = 0; i < NL; i++)
            __builtin_amdgcn_global_load_lds((global_ptr_t) ((i * RPL < BC ? abase : bbase) + at + (last ? off_last[i] : off[i])), (lds_ptr_t) (ring + stage * STAGE + i * 1024), 16, 0, 0);
    };
    vec av[SEG / 4][MB], bv[SEG / 4][NB];
    // NORM: the normalised rows, a vector further apart than they are long (a piece of the last may end behind it: that is cleared)
    T* const normed = reinterpret_cast<T*>(waves_lds + NW * STAGES * STAGE);
    const int pitch = (int) k + VK;
    auto read = [&](int piece, int stage) {
#pragma unroll
        for (int h = 0; h < SEG / 4; h++) {
#pragma unroll
            for (int i = 0; i < MB + NB; i++) {
                const int row = (i < MB ? i : i - MB) * 16 + idx;
                if (NORM && i < MB) {
                    av[h][i] = *reinterpret_cast<const vec*>(normed + row % MR * pitch + piece * PIECE + (h * 4 + grp) * VK);
                } else {
                    const vec v = *reinterpret_cast<const vec*>(ring + stage * STAGE + ((i < MB ? 0 : BC) + row) * (SEG * 16) + ((h * 4 + grp) ^ swz(row)) * 16);
                    if (i < MB) av[h][i] = v;
                    else bv[h][i - MB] = v;
                }
            }
        }
    };
    auto clear = [&]() {
#pragma unroll
        for (int h = 0; h < SEG / 4; h++) {
            const bool in = (h * 4 + grp) * VK < kleft;
#pragma unroll
            for (int i = 0; i < MB; i++) av[h][i] = in ? av[h][i] : vec{};
#pragma unroll
            for (int j = 0; j < NB; j++) bv[h][j] = in ? bv[h][j] : vec{};
        }
    };
    // (operands swapped: a lane has four consecutive columns of a row)
    f32x4 acc[SUMS][MB][NB];
#pragma unroll
    for (int u = 0; u < SUMS; u++)
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < NB; j++) acc[u][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](auto odd_c) {      // odd: every other piece of a wavefront
        constexpr int ODD = decltype(odd_c)::value;
#pragma unroll
        for (int h = 0; h < SEG / 4; h++) {
            if constexpr (F32) {
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int i = 0; i < MB; i++)
#pragma unroll
                        for (int j = 0; j < NB; j++) acc[(ODD * 4 + e) % SUMS][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[h][j][e], av[h][i][e], acc[(ODD * 4 + e) % SUMS][i][j], 0, 0, 0);
            } else {
#pragma unroll
                for (int i = 0; i < MB; i++)
#pragma unroll
                    for (int j = 0; j < NB; j++) acc[(ODD * 2 + h) % SUMS][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bv[h][j], av[h][i], acc[(ODD * 2 + h) % SUMS][i][j], 0, 0, 0);
            }
        }
    };
    // this wavefront's pieces: wave, wave + NW, ...
    const int mine_n = pieces > wave ? (pieces - wave + NW - 1) / NW : 0;
    auto start = [&]() {
#pragma unroll
        for (int s = 0; s < STAGES; s++)
            if (s < mine_n) copy(wave + s * NW, s);
    };
    if constexpr (NORM > 0) {
        // the rows and the norm's operands first: loads arrive in the order they were issued in
        constexpr int RPW = (MR + NW - 1) / NW;
        vec x[RPW][NORM], w[NORM], b[NORM];
        const int vectors = (int) k / VK;
        auto at = [&](int i) { return i * 64 + lane < vectors ? (i * 64 + lane) * VK : 0; };
#pragma unroll
        for (int r = 0; r < RPW; r++)
#pragma unroll
            for (int i = 0; i < NORM; i++) x[r][i] = *reinterpret_cast<const vec*>(A + (r * NW + wave < m ? r * NW + wave : 0) * lda + at(i));
#pragma unroll
        for (int i = 0; i < NORM; i++) {
            if (norm.weight) w[i] = *reinterpret_cast<const vec*>(reinterpret_cast<const T*>(norm.weight) + at(i));
            if (norm.bias) b[i] = *reinterpret_cast<const vec*>(reinterpret_cast<const T*>(norm.bias) + at(i));
        }
        __builtin_amdgcn_sched_barrier(0);
        start();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < RPW; r++) {
            float v[NORM][VK], sum = 0.f, sq = 0.f;
#pragma unroll
            for (int i = 0; i < NORM; i++)
#pragma unroll
                for (int e = 0; e < VK; e++) {
                    v[i][e] = i * 64 + lane < vectors ? (float) x[r][i][e] : 0.f;
                    sum += v[i][e];
                }
            const float mean = wave_sum(sum) / (float) k;
#pragma unroll
            for (int i = 0; i < NORM; i++)
#pragma unroll
                for (int e = 0; e < VK; e++) {
                    v[i][e] -= mean;
                    if (i * 64 + lane < vectors) sq += v[i][e] * v[i][e];
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
                if (r * NW + wave < MR && i * 64 + lane < vectors)
                    *reinterpret_cast<vec*>(normed + (r * NW + wave) * pitch + (i * 64 + lane) * VK) = r * NW + wave < m ? out : vec{};
            }
        }
        // (not __syncthreads: that would wait for the copies)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    } else {
        start();
    }
    auto step = [&](int i, int stage, auto odd_c) {
        const int piece = wave + i * NW, newer = mine_n - 1 - i;
        // the stage has landed once no more than the copies of the newer ones are on their way
        if (newer >= STAGES - 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 1) * NL) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        read(piece, stage);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // the stage is read: its place is free
        if (i + STAGES < mine_n) copy(piece + STAGES * NW, stage);
        if (kleft < PIECE && piece == pieces - 1) clear();
        multiply(odd_c);
    };
    static_assert(STAGES == 2, "a pair of pieces an iteration");
    for (int i = 0; i < mine_n; i += 2) {
        step(i, 0, std::integral_constant<int, 0>{});
        if (i + 1 < mine_n) step(i + 1, 1, std::integral_constant<int, 1>{});
    }
#pragma unroll
    for (int u = SUMS / 2; u >= 1; u /= 2)
#pragma unroll
        for (int q = 0; q < u; q++)
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int j = 0; j < NB; j++) acc[q][i][j] += acc[q + u][i][j];
    __syncthreads();     // the rings end here

    float* const sums = reinterpret_cast<float*>(waves_lds);
    float* const mine = sums + (wave % COPIES) * (BM * LDW);
    auto each = [&](auto use) {
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < NB; j++) use(acc[0][i][j], reinterpret_cast<f32x4*>(mine + (i * 16 + idx) * LDW + j * 16 + (lane >> 4) * 4));
    };
    if constexpr (TWICE) {
        if (wave >= COPIES) each([](f32x4& a, f32x4* at) { *at = a; });
        __syncthreads();
        // (a lane's own words: no barrier between the two)
        if (wave < COPIES) each([](f32x4& a, f32x4* at) { *at = a + *at; });
    } else {
        each([](f32x4& a, f32x4* at) { *at = a; });
    }
    __syncthreads();
    constexpr int UPR = BN / 8;
#pragma unroll 1
    for (int unit = tid; unit < BM * UPR; unit += 64 * NW) {
        const int t = unit / UPR, c8 = unit % UPR * 8;
        if (t < rows && c8 < cols) {
            float v[8], b[8];
            f32x4 lo{}, hi{};
#pragma unroll
            for (int w = 0; w < COPIES; w++) {
                const f32x4* from = reinterpret_cast<const f32x4*>(sums + w * (BM * LDW) + t * LDW + c8);
                lo += from[0], hi += from[1];
            }
#pragma unroll
            for (int e = 0; e < 8; e++) {
                v[e] = alpha * (e < 4 ? lo[e & 3] : hi[e & 3]);
                asm volatile("" : "+v"(v[e]));    // the product is rounded before the bias is added
                b[e] = -0.0f;
            }
            if (f.bias) load8(f.bias, n0 + c8, f.flags & kBiasBf16, b);
            finish8(f, v, b, (m0 + t) * n + n0 + c8);
        }
    }
}

} // namespace docc_k

#define DOCC_GEMM_WAVES(NAME, T, BM, BN, NW, SEG, SUMS, PER_CU)                                                                                                \
    extern "C" __global__ __launch_bounds__(64 * NW, NW * PER_CU / 4) void NAME(const T* A, long lda, const T* B, long ldb, long m, long n, long k, float alpha, \
                                                                                docc_k::GemmFinish f) {                                                       \
        docc_k::gemm_waves<T, BM / 16, BN / 16, NW, SEG, 2, SUMS, 0, 0>(A, lda, B, ldb, m, n, k, alpha, f, docc_k::RowsNorm{});                               \
    }
DOCC_GEMM_WAVES(docc_bgemm_waves_16x16_f, uint16_t, 16, 16, 8, 8, 4, 2)
DOCC_GEMM_WAVES(docc_sgemm_waves_16x16_f, float, 16, 16, 8, 8, 4, 2)
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
        docc_k::gemm_waves<T, 1, 1, 8, 8, 2, 4, L, R>(X, ldx, B, ldb, m, n, k, alpha, f, norm);                                                               \
    }
DOCC_GEMM_WAVES_NORM(b, uint16_t, 8, 4, 2)
DOCC_GEMM_WAVES_NORM(b, uint16_t, 8, 8, 1)
DOCC_GEMM_WAVES_NORM(b, uint16_t, 16, 4, 1)
DOCC_GEMM_WAVES_NORM(s, float, 8, 4, 2)
DOCC_GEMM_WAVES_NORM(s, float, 8, 8, 2)
DOCC_GEMM_WAVES_NORM(s, float, 16, 4, 2)
