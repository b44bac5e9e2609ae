// A product, or a layer, on few rows, or any that has too few tiles to fill the compute units: out = finish(alpha * A[m, k] B[n][k]^T), the chain of gemm_finish.h behind
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
#pragma once

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
//
// B is stored [n][k], or with TB false [k][n]: then a piece is PIECE of its rows as far as the tile goes.
template <typename T, int MB, int NB, int NW, int SEG, int STAGES, int SUMS, int NORM, int MR, bool TB, typename Store>
__device__ __forceinline__ void gemm_waves(const T* __restrict__ A, long lda, const T* __restrict__ B, long ldb, long m, long n, long k, const Store& out, const RowsNorm& norm) {
    constexpr bool F32 = sizeof(T) == 4, F64 = sizeof(T) == 8;
    typedef std::conditional_t<F64, double, float> S;
    constexpr int VK = 16 / (int) sizeof(T), PIECE = SEG * VK, BM = 16 * MB, BN = 16 * NB, LDW = BN + 16 / (int) sizeof(S);
    constexpr int BC = NORM ? 0 : BM;      // rows of A that are copied
    constexpr int STAGE = (BC + BN) * SEG * 16, NL = (BC + BN) * SEG / 64, RPL = 64 / SEG;    // bytes, copies and a copy's rows of a stage
    constexpr bool TWICE = NW * BM * LDW * (int) sizeof(S) > 65536;      // the sums of half of the wavefronts at a time
    constexpr int COPIES = TWICE ? NW / 2 : NW;
    static_assert((SEG == 4 || SEG == 8) && (STAGES - 1) * NL < 64, "the swizzles; vmcnt holds at most 63 outstanding copies");
    static_assert(SUMS == 1 || (F32 ? (SUMS == 16 && SEG == 8) || SUMS == 8 || SUMS == 4 || SUMS == 2 : SUMS == 2 || (SUMS == 4 && SEG == 8)), "a product's set is known at compile time");
    static_assert(NORM == 0 || (MB == 1 && MR <= 16), "the rows that are normalised");
    typedef std::conditional_t<F64, f64x2, std::conditional_t<F32, f32x4, bf16x8>> vec;
    typedef std::conditional_t<F64, f64x4, f32x4> sum4;
    extern __shared__ __attribute__((aligned(16))) unsigned char waves_lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int idx = lane & 15, grp = lane >> 4;
    int tm, tn;
    gemm_tile_coords(blockIdx.x, (int) ((m + BM - 1) / BM), (int) ((n + BN - 1) / BN), tm, tn);
    const long m0 = (long) tm * BM, n0 = (long) tn * BN;
    const int rows = m - m0 < BM ? (int) (m - m0) : BM, cols = n - n0 < BN ? (int) (n - n0) : BN;
    const int pieces = (int) ((k + PIECE - 1) / PIECE), kleft = (int) (k - (long) (pieces - 1) * PIECE);   // k of the last piece
    auto swz = [](int row) { return SEG == 8 ? row & 7 : (row >> 2) & 3; };
    // [k][n]: granules across the tile, XORed so that the four groups of lanes, which read different rows, meet in few banks
    constexpr int GPR = BN * (int) sizeof(T) / 16;
    auto swz_n = [](int kr) {
        if constexpr (F64) return GPR >= 16 ? ((kr >> 1) & 1) * 8 : 0;
        else if constexpr (F32) return GPR == 16 ? ((kr >> 2) & 3) * 4 : GPR == 8 ? ((kr >> 2) & 1) * 4 : 0;
        else return GPR == 8 ? 2 * (((kr >> 1) & 1) | ((kr >> 3) & 1) << 1) : GPR == 4 ? 2 * ((kr >> 3) & 1) : 0;
    };

    // copy i of a stage: rows RPL i .. of the tile's BM + BN, those beyond the edge as copies of the last (their products are not stored)
    unsigned off[NL], off_last[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const bool is_a = i * RPL < BC;
        if (!TB && !is_a) {
            const int g = (i * RPL - BC) * SEG + lane, kr = g / GPR, col = (g % GPR ^ swz_n(kr)) * VK;
            const int c = col < cols ? col : cols - VK;       // (whole granules: n is a multiple of VK)
            off[i] = (unsigned) kr * (unsigned) (ldb * (long) sizeof(T)) + c * (int) sizeof(T);
            off_last[i] = kr < kleft ? off[i] : c * (int) sizeof(T);
            continue;
        }
        const int row = (is_a ? i * RPL : i * RPL - BC) + lane / SEG, granule = (lane % SEG) ^ swz(row);
        const int r = is_a ? (row < rows ? row : rows - 1) : (row < cols ? row : cols - 1);
        off[i] = (unsigned) r * (unsigned) ((is_a ? lda : ldb) * (long) sizeof(T)) + granule * 16;
        off_last[i] = off[i] - (granule * VK < kleft ? 0 : granule * 16);     // behind the end of K: the first of the row, cleared in registers
    }
    const char* const abase = reinterpret_cast<const char*>(A + m0 * lda);
    const char* const bbase = reinterpret_cast<const char*>(TB ? B + n0 * ldb : B + n0);
    unsigned char* const ring = waves_lds + wave * (STAGES * STAGE);
    auto copy = [&](int piece, int stage) {
        const long at = (long) piece * (16 * SEG), bat = TB ? at : (long) piece * PIECE * ldb * (long) sizeof(T);
        const bool last = piece == pieces - 1;
#pragma unroll
        for (int i = 0; i < NL; i++)
            __builtin_amdgcn_global_load_lds((global_ptr_t) ((i * RPL < BC ? abase + at : bbase + bat) + (last ? off_last[i] : off[i])), (lds_ptr_t) (ring + stage * STAGE + i * 1024), 16, 0, 0);
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
                if (!TB && i >= MB) {
                    unsigned char* const at = ring + stage * STAGE + BC * SEG * 16;
                    const int j0 = (i - MB) * 16;
                    if constexpr (F32 || F64) {
#pragma unroll
                        for (int e = 0; e < VK; e++) {
                            const int kr = (h * 4 + grp) * VK + e, col = j0 + idx;
                            bv[h][i - MB][e] = *reinterpret_cast<const T*>(at + kr * (BN * (int) sizeof(T)) + ((col / VK) ^ swz_n(kr)) * 16 + (col % VK) * (int) sizeof(T));
                        }
                    } else {
                        // transposed reads: 16 lanes give the addresses of four rows of 16 columns and get four k of a column each
                        const int kr = (h * 4 + grp) * 8 + (idx >> 2), col = j0 + 4 * (idx & 3);
                        typedef __attribute__((address_space(3))) s16x4a lds_s16x4;
                        const s16x4a lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*) (at + kr * (BN * 2) + ((col / 8) ^ swz_n(kr)) * 16 + (col % 8) * 2));
                        const s16x4a hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*) (at + (kr + 4) * (BN * 2) + ((col / 8) ^ swz_n(kr + 4)) * 16 + (col % 8) * 2));
                        const s16x8a v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                        bv[h][i - MB] = __builtin_bit_cast(bf16x8, v);
                    }
                } else if (NORM && i < MB) {
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
    sum4 acc[SUMS][MB][NB];
#pragma unroll
    for (int u = 0; u < SUMS; u++)
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < NB; j++) acc[u][i][j] = sum4{};
    auto multiply = [&](auto odd_c) {      // odd: every other piece of a wavefront
        constexpr int ODD = decltype(odd_c)::value;
#pragma unroll
        for (int h = 0; h < SEG / 4; h++) {
            if constexpr (F64) {
#pragma unroll
                for (int e = 0; e < 2; e++)
#pragma unroll
                    for (int i = 0; i < MB; i++)
#pragma unroll
                        for (int j = 0; j < NB; j++) acc[e % SUMS][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[h][j][e], av[h][i][e], acc[e % SUMS][i][j], 0, 0, 0);
            } else if constexpr (F32) {
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int i = 0; i < MB; i++)
#pragma unroll
                        for (int j = 0; j < NB; j++) acc[((SUMS == 16 ? h * 8 : 0) + ODD * 4 + e) % SUMS][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[h][j][e], av[h][i][e], acc[((SUMS == 16 ? h * 8 : 0) + ODD * 4 + e) % SUMS][i][j], 0, 0, 0);
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

    S* const sums = reinterpret_cast<S*>(waves_lds);
    S* const mine = sums + (wave % COPIES) * (BM * LDW) + idx * LDW + (F64 ? grp : 4 * grp);
    auto each = [&](auto use) {
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < NB; j++) {
                S* const at = mine + i * 16 * LDW + j * 16;
                if constexpr (F64) {      // register r: column 4 r + grp
#pragma unroll
                    for (int r = 0; r < 4; r++) use(acc[0][i][j][r], at + 4 * r);
                } else {
                    use(acc[0][i][j], reinterpret_cast<f32x4*>(at));
                }
            }
    };
    if constexpr (TWICE) {
        if (wave >= COPIES) each([](auto a, auto* at) { *at = a; });
        __syncthreads();
        // (a lane's own words: no barrier between the two)
        if (wave < COPIES) each([](auto a, auto* at) { *at = a + *at; });
    } else {
        each([](auto a, auto* at) { *at = a; });
    }
    __syncthreads();
    out.template store<BM, BN, LDW, COPIES, 64 * NW>(sums, tid, m0, n0, rows, cols, n);
}

// the wavefronts' sums in pairs: fewer roundings than one after the other (with that a matrix-vector product stays as exact as the kernels of gemv.hip)
template <int COPIES, typename V, typename F>
__device__ __forceinline__ V waves_sum(F part) {
    V v[COPIES];
#pragma unroll
    for (int w = 0; w < COPIES; w++) v[w] = part(w);
#pragma unroll
    for (int u = COPIES / 2; u >= 1; u /= 2)
#pragma unroll
        for (int q = 0; q < u; q++) v[q] += v[q + u];
    return v[0];
}

// the chain of a layer: a lane finishes eight consecutive columns of a row
struct WavesFinish {
    GemmFinish f;
    float alpha;
    template <int BM, int BN, int LDW, int COPIES, int THREADS>
    __device__ __forceinline__ void store(const float* sums, int tid, long m0, long n0, int rows, int cols, long n) const {
        constexpr int UPR = BN / 8;
#pragma unroll 1
        for (int unit = tid; unit < BM * UPR; unit += THREADS) {
            const int t = unit / UPR, c8 = unit % UPR * 8;
            if (t < rows && c8 < cols) {
                float v[8], b[8];
                const float* from = sums + t * LDW + c8;
                const f32x4 lo = waves_sum<COPIES, f32x4>([&](int w) { return *reinterpret_cast<const f32x4*>(from + w * (BM * LDW)); });
                const f32x4 hi = waves_sum<COPIES, f32x4>([&](int w) { return *reinterpret_cast<const f32x4*>(from + w * (BM * LDW) + 4); });
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
};

// C = alpha A B + beta C, lanes along the columns
template <typename S>
struct WavesPlain {
    S* C;
    long ldc;
    S alpha, beta;
    const S* bias;     // one value per column, or null
    int act;           // abs, relu or -1
    template <int BM, int BN, int LDW, int COPIES, int THREADS>
    __device__ __forceinline__ void store(const S* sums, int tid, long m0, long n0, int rows, int cols, long) const {
        const int c = tid % BN;
        if (c >= cols) return;
        S* const to = C + m0 * ldc + n0 + c;
        constexpr int STEP = THREADS / BN;
        static_assert(THREADS % BN == 0, "a lane keeps its column");
        auto sum = [&](int t) { return waves_sum<COPIES, S>([&](int w) { return sums[w * (BM * LDW) + t * LDW + c]; }); };
        const S b = bias ? bias[n0 + c] : (S) -0.0;
        auto finish = [&](S val) {
            asm volatile("" : "+v"(val));   // the product is rounded before the bias is added, as by the separate nodes
            val += b;
            return act == kReLU ? unary<kReLU>(val) : act == kAbs ? unary<kAbs>(val) : val;
        };
        if (beta == (S) 0) {
#pragma unroll 4
            for (int t = tid / BN; t < rows; t += STEP) to[t * ldc] = finish(alpha * sum(t));
        } else {
#pragma unroll 4
            for (int t = tid / BN; t < rows; t += STEP) to[t * ldc] = finish(gemm_axpby(alpha, sum(t), beta, to[t * ldc]));
        }
    }
};

} // namespace docc_k
