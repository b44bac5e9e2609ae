// Launchers for the GEMM node kernels (see include/docc_rocm_ops.h).
#include <cstdio>
#include <type_traits>
#include <cstdlib>
#include <cstring>

#include "docc_rocm_ops.h"
#include "rt_state.h"

using namespace docc::rt::rocm;

namespace {

struct TileConfig {
    int bm, bn, bk, waves;
    int stages;  // > 0: asynchronous multi-stage kernel (gemm_async.h), aligned operands only
    bool spread = false;  // asynchronous kernels: the variant that deals a stage's copies over the whole K-step (3 stages or more)
    bool small = false;   // asynchronous bf16 kernels: the variant built on the 16x16x32 MFMA
};

// LDS bytes of GemmKernel<T, BM, BN, BK, ...> (csrc/kernels/gemm_mfma.h)
size_t gemm_lds_bytes(const TileConfig& c, bool ta, bool tb, size_t elem) {
    // fp32/fp64 pad mn-contiguous rows by 8 elements, bf16 (GemmBf16Kernel) by 16
    const int padk = (int) (16 / elem), padm = elem == 2 ? 16 : 8;
    const bool a_kc = !ta, b_kc = tb;
    const int lda_s = a_kc ? c.bk + padk : c.bm + padm;
    const int ldb_s = b_kc ? c.bk + padk : c.bn + padm;
    const size_t a_elems = (size_t) (a_kc ? c.bm : c.bk) * lda_s;
    const size_t b_elems = (size_t) (b_kc ? c.bn : c.bk) * ldb_s;
    return 2 * (a_elems + b_elems) * elem;
}

// Seconds a bf16 product of `count` matrices takes on tile `c`, fitted to 440 drawn products (64 to 8192 an extent, on and off whole lines,
// a third with an epilogue) on all four tiles: a launch, and for every round of tiles over the CUs the fp32 store of the tiles (all of them at
// once: 11 us for 256 x 256) and their products at what the tile sustains. A last round that leaves CUs idle runs faster (less traffic, higher
// clocks), but not in proportion. The 128 x 128 tile with stages of 32 k sits two to a CU: 264 of them are little more than one round, where the
// others need a second (1509 x 2816 x 1032: 22 us, the one with stages of 64 k 28, 128 x 256 26). `lines`: the operands' rows start on lines of
// 128 bytes; a stage of 64 k that does not straddles two. On 660 other products the tile that this estimate takes is 0.8 % slower than the
// fastest in the mean and more than 5 % on 33 of them; by the number of 256 x 256 tiles alone (from 192 on that tile, else 128 x 128 with
// stages of 32 k) it is 5.0 % and 171.
double bgemm_seconds(const TileConfig& c, int64_t m, int64_t n, int64_t k, bool tb, int64_t count, int cus, bool lines) {
    const bool big = c.bm == 256, wide = c.bm < c.bn, two = !big && !wide && c.bk == 32, pairs = k % 64 == 0;   // pairs: K as the 16x16x32 MFMA takes it
    const int64_t tiles = ((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn) * count, round = two ? 2 * cus : cus, last = tiles % round;
    const double part = (double) last / cus;
    double rounds = (double) (tiles / round) * (two ? 1.44 : 1.0);
    if (last) rounds += !two ? 0.66 + 0.37 * part : part <= 1.0 ? 0.41 + 0.33 * part : 0.68 + 0.38 * part;
    if (!big && !wide && !two && tiles <= cus) rounds = 0.56 + 0.3 * (double) tiles / cus;
    // relative to the 256 x 256 tile: the 128 x 256 one reads a k-major B from LDS at half the width; 128 x 128 tiles wait for their copies
    double rel = big ? (pairs ? 1.0 : 0.88) : wide ? (tb ? 0.75 : 0.71) : two ? 0.44 : tiles > cus ? 0.68 : 0.61;
    if (!lines) rel *= big ? (pairs ? 0.95 : 1.0) : wide ? 0.88 : 0.85;
    const double area = (double) c.bm * c.bn, fill = big ? (pairs ? 1.0 : 2.0) : wide || two ? 0.0 : 0.4;   // us until a round's first products
    return 1e-6 * (4.0 + rounds * (fill + area * (11.0 / 65536) + area * (double) k * 3.6e-7 / rel));
}

// The same for an fp32 or fp64 product (`k`: of all its `parts` together): the work of the padded tiles at what the tile sustains (relative to the
// 128 x 256 one), on the share of the CUs' time that does work: below one work-group per CU the CUs that get one, above it the whole
// rounds (344 work-groups on 256 CUs take as long as 512).
double sdgemm_seconds(const TileConfig& c, int64_t m, int64_t n, int64_t k, int64_t parts, int cus, size_t elem) {
    const double tm = (double) ((m + c.bm - 1) / c.bm), tn = (double) ((n + c.bn - 1) / c.bn);
    const double area = (double) c.bm * c.bn, rel = area >= 65536 ? 1.03 : area >= 32768 ? 1.0 : area >= 16384 ? 0.97 : 0.75;
    const double per_cu = tm * tn * (double) parts / cus, fill = per_cu < 1.0 ? per_cu : per_cu / (double) (int64_t) (per_cu + 0.999999);
    return 2.0 * tm * c.bm * tn * c.bn * (double) k / ((elem == 8 ? 68e12 : 141e12) * rel * fill);
}

using Picker = TileConfig (*)(int64_t m, int64_t n, int64_t k, bool tb, int64_t batch, int aligned, int force, int cus);

constexpr int64_t kMaxPartsBytes = int64_t(64) << 20;   // of the parts of a product whose K is cut
constexpr int64_t kPartCounts[] = {2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32, 48, 64};
// k of a part: whole steps of 64 of every tile; the last part takes what is left
int64_t part_length(int64_t k, int64_t parts) { return ((k + parts - 1) / parts + 63) / 64 * 64; }

// ... and with K in the best number of parts, as gemm_launch cuts it (below)
double sdgemm_best_seconds(Picker pick, int64_t m, int64_t n, int64_t k, bool tb, int cus, size_t elem) {
    const TileConfig whole = pick(m, n, k, tb, 1, 2, 0, cus);
    double best = sdgemm_seconds(whole, m, n, k, 1, cus, elem);
    if (k < 512 || ((m + whole.bm - 1) / whole.bm) * ((n + whole.bn - 1) / whole.bn) >= cus) return best;
    for (const int64_t parts : kPartCounts) {
        const int64_t part = part_length(k, parts), bytes = parts * m * n * (int64_t) elem;
        if ((k + part - 1) / part != parts || part < 256 || bytes > kMaxPartsBytes) continue;
        const double t = sdgemm_seconds(pick(m, n, part, tb, parts, 2, 0, cus), m, n, k, parts, cus, elem) + 2.0 * (double) bytes / 5e12 + 3e-6;
        if (t < best) best = t;
    }
    return best;
}

// Seconds of a product on the tiles, whole or in parts (the pass that adds them counted)
double tiles_seconds(Picker pick, int64_t m, int64_t n, int64_t k, bool tb, int cus, size_t elem, bool lines) {
    if (elem != 2) return 4.0e-6 + sdgemm_best_seconds(pick, m, n, k, tb, cus, elem);
    const TileConfig whole = pick(m, n, k, tb, 1, lines ? 2 : 1, 0, cus);
    double best = bgemm_seconds(whole, m, n, k, tb, 1, cus, lines);
    if (k < 512 || ((m + whole.bm - 1) / whole.bm) * ((n + whole.bn - 1) / whole.bn) >= cus) return best;
    for (const int64_t parts : kPartCounts) {
        const int64_t part = part_length(k, parts), bytes = parts * m * n * 4;
        if ((k + part - 1) / part != parts || part < 256 || bytes > kMaxPartsBytes) continue;
        const double t = bgemm_seconds(pick(m, n, part, tb, parts, lines ? 2 : 1, 0, cus), m, n, part, tb, parts, cus, lines) + 2.0 * (double) bytes / 5e12 + 3.5e-6;
        if (t < best) best = t;
    }
    return best;
}

// The tile of csrc/kernels/gemm_waves.hip and its estimate: a launch, and so long a tile on the compute unit that has most of them. Fitted to 58 products a type from
// 33 x 64 x 256 to 4096 x 2048 x 512, of most of them less than 10 % off.
struct WavesChoice {
    int edge;
    bool one;        // no compute unit has two
    double seconds;
};
// `lines`: rows of both operands are whole lines of 128 bytes. Off them a piece of a row takes two lines, which for fp32 and fp64 on 16 x 16 tiles (the least work a byte)
// are no longer in the caches when the next piece wants them: fp64 581 x 194 x 2322 1.35 times the estimate, 266 x 1411 x 3730 1.55, 968 x 183 x 5886 1.62, with a tile a
// compute unit from 4300 k on; fp32 1130 x 262 x 5032 1.35, 1880 x 137 x 6228 1.49. bf16 on its larger tiles once they read more than so many bytes in all: of 32 x 32 175
// MB (581 x 752 x 4184 1.5, 499 x 728 x 7064 1.52; with 164, 162 x 2208 x 3096, 1.0), of 64 x 64 120 MB (1664 x 560 x 2536 1.59, 596 x 2664 x 3880 1.8; with 101, 98 x 6776 x
// 1864, 1.0), on the lines 400 MB in rows of more than 3000 k (644 x 5696 x 4416 1.28, 262 x 6016 x 3904 1.24). fp32 and fp64 on those no different.
WavesChoice waves_choice(int64_t m, int64_t n, int64_t k, int cus, size_t elem, bool lines, int forced) {
    auto per_cu = [&](int64_t edge) { return (double) ((((m + edge - 1) / edge) * ((n + edge - 1) / edge) + cus - 1) / cus); };
    const double n16 = per_cu(16), n32 = per_cu(32), n64 = per_cu(64), kd = (double) k;
    const bool one = n64 <= 1.0 && (elem == 4 || k > 1024);
    const double straddle = lines || elem == 2 ? 1.0 : elem == 4 ? (n16 <= 1.0 ? 1.0 : k < 7800 ? 1.0 + kd / 13000.0 : 1.6)
                            : n16 > 1.0 ? (k < 5400 ? 1.0 + kd / 9000.0 : 1.6) : k < 4300 ? 1.0 : 1.4;
    const double t16 = elem == 2 ? 3.8 + n16 * (0.4 + 0.00065 * kd) : elem == 4 ? 4.0 + n16 * (0.5 + 0.00125 * straddle * kd) : 3.8 + n16 * (0.6 + 0.0024 * straddle * kd);
    auto reads_mb = [&](int64_t edge) { return 1e-6 * (double) (((m + edge - 1) / edge) * ((n + edge - 1) / edge)) * 4.0 * (double) edge * kd; };
    const double far32 = !lines && reads_mb(32) > 175.0 ? 1.5 : 1.0, far64 = lines ? (k > 3000 && reads_mb(64) > 400.0 ? 1.25 : 1.0) : reads_mb(64) > 120.0 ? 1.5 : 1.0;
    const double t32 = elem == 2 ? 3.4 + n32 * (0.75 + 0.0010 * far32 * kd) : elem == 4 ? 3.7 + n32 * (0.75 + 0.0043 * kd) : 3.8 + n32 * (0.9 + 0.0092 * kd);
    const double t64 = elem == 2 ? (one ? 4.75 + 0.0028 * far64 * kd : 1.9 + n64 * (2.1 + 0.0027 * far64 * kd))
                                 : 3.7 + n64 * (1.2 + 0.0172 * kd);
    if (forced > 0 ? forced == 16 : m <= 16 || (t16 < t32 && (elem == 8 || t16 < t64))) return {16, false, 1e-6 * t16};
    // (fp64: 64 x 64 tiles of 1000 k took 39.0 us for the 37.0 of gemm_async.h's)
    if (elem == 8 || (forced > 0 ? forced == 32 : t32 <= t64)) return {32, false, 1e-6 * t32};
    return {64, forced > 0 ? forced == 1 : one, 1e-6 * t64};
}
// what the kernels read: whole vectors, a tile's rows within 32 bits of its first
bool waves_shape_ok(int64_t m, int64_t n, int64_t k, int64_t lda, int64_t ldb, bool tb, size_t elem) {
    const int64_t v = 16 / (int64_t) elem, lim = (int64_t(1) << 25) / (int64_t) elem;
    return k > 0 && k % v == 0 && lda % v == 0 && ldb % v == 0 && (tb || n % v == 0) && k < lim && lda < lim && ldb < lim && m < (int64_t(1) << 24) && n < (int64_t(1) << 24) &&
           ((m + 15) / 16) * ((n + 15) / 16) < (int64_t(1) << 31);
}

// Microseconds of an fp32 or fp64 product on the element-wise tiles (operands off the vectors): a round of tiles over the CUs takes so long per k.
// `turned`: an operand is read along m or n.
double plain_us(Picker pick, int64_t m, int64_t n, int64_t k, bool tb, bool turned, int cus, size_t elem) {
    const TileConfig c = pick(m, n, k, tb, 1, 0, 0, cus);
    const int64_t tiles = ((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn), rounds = (tiles + cus - 1) / cus;
    const double first = elem == 8 ? (turned ? 0.006 : 0.008) : c.bm == 64 ? (turned ? 0.015 : 0.0045) : turned ? 0.0 : 0.01;
    const double each = elem == 8 ? (turned ? 0.036 : 0.0345) : c.bm == 64 ? (turned ? 0.0172 : 0.0165) : turned ? 0.08 : 0.065;
    return 5.0 + (double) k * (first + each * (double) rounds);
}

// the number of CUs, asked for once per call of an entry point: a product with fewer tiles than CUs weighs up to 60 forms by it
int cu_count() {
    const int cus = compute_units();
    return cus > 0 ? cus : 256;
}

// What GemmFinish of csrc/kernels/gemm_finish.h holds: the rest of a layer behind a product.
struct LinearFinish {
    const void *bias, *residual;
    void* out;
    int flags, act;
};
enum { kBiasBf16 = 1, kResidualBf16 = 2, kOutBf16 = 4, kRoundBeforeAct = 8, kRoundAfterAct = 16 };

// the chain on `parts` fp32 products in memory
int finish_parts(hipStream_t s, const void* P, int64_t m, int64_t n, int parts, float alpha, const LinearFinish& f) {
    const bool vec = n % 8 == 0 && ((uintptr_t) P | (uintptr_t) f.bias | (uintptr_t) f.residual | (uintptr_t) f.out) % 16 == 0;
    const int64_t units = m * n / (vec ? 8 : 1);
    int64_t blocks = (units + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    return launch(vec ? "docc_gemm_finish_v8" : "docc_gemm_finish_v1", (uint32_t) blocks, 1, 1, 256, 0, s, P, (long) m, (long) n, parts, alpha, f);
}

// One output column or one output row: the matrix-vector kernels (csrc/kernels/gemv.hip). Returns 1 when the
// shape is not one of theirs (the caller goes on to the tiled kernels), 0 or an error code otherwise.
template <typename T, typename S>
int gemv_launch(const char* prefix, hipStream_t s, bool ta, bool tb, int64_t m, int64_t n, int64_t k, S alpha, const T* A, int64_t lda,
                const T* B, int64_t ldb, S beta, S* C, int64_t ldc, bool tuned, int cus) {
    if (tuned && std::getenv("DOCC_ROCM_GEMV_OFF")) return 1;   // tuning and tests: always the tiled kernels
    const T *M, *x;
    int64_t ld, incx, incy, rows, cols;
    bool by_rows;
    if (m > 1 && n > 1) {
        // two to eight rows or columns of output with both operands stored row by row along k (op(A) = A, op(B) = B^T,
        // the product of a small batch with a weight matrix): the larger operand moves once
        if (m > 8 && n > 8) return 1;
        // five to eight vectors would be two passes over the matrix: the tiles with K in parts are faster (fp32 8 x 4096 x 4096:
        // 39 us here, 26 there; 8 x 8192 x 8192: 95 against 81; fp64 8 x 8192 x 8192: 296 against 172)
        const int64_t max_vectors = 4;
        if (sizeof(T) != 2 && ((m <= max_vectors && !ta && !tb) || (n <= max_vectors && ta && !tb && m > 8))) {
            // the large operand is stored [k][columns] (y = x W with W as numpy holds it): columns form, sliced over k
            const bool small_a = m <= max_vectors && !ta;
            const int64_t nv = small_a ? m : n, cols = small_a ? n : m;
            const T* mat = small_a ? B : A;
            const T* vecs = small_a ? A : B;
            const int64_t ldm = small_a ? ldb : lda;
            const int64_t sx_v = small_a ? lda : 1, sx_p = small_a ? 1 : ldb;          // A[v][p] or B[p][v]
            const int64_t sy_vec = small_a ? ldc : 1, sy_col = small_a ? 1 : ldc;
            if (cols < 1024 || k < 64) return 1;
            const int vecw = 16 / (int) sizeof(T);
            const bool aligned = (uintptr_t) mat % 16 == 0 && ldm % vecw == 0 && cols % vecw == 0;
            const int lanes = aligned ? vecw : 1;
            const int64_t col_blocks = (cols / lanes + 255) / 256;
            // 1.75 work-groups per CU (measured against 0.75 .. 6 per CU on five shapes: 4 x 8192 x 8192 in 46.9 us against
            // 51.7 with two, 8 x 8192 x 8192 in 93.9 against 102.3, 4 x 4096 x 11008 in 32.9 against 35.3)
            int64_t slices = (7 * (int64_t) cus / 4 + col_blocks - 1) / col_blocks;
            if (slices > k / 16) slices = k / 16;
            // the partial sums are written and read back: keep them under a sixteenth of the matrix's bytes
            const int64_t group = nv < 4 ? nv : 4;                                     // vectors per pass
            int64_t cheap = k * (int64_t) sizeof(T) / (16 * (int64_t) sizeof(S) * group);
            if (cheap * col_blocks < 4 * (int64_t) cus) cheap *= 2;      // ... unless that leaves the chip short of work-groups
            if (slices > cheap) slices = cheap;
            const int64_t fit = (int64_t) kPartialsBytes / ((int64_t) sizeof(S) * cols * group);
            if (slices > fit) slices = fit;
            if (slices > 256) slices = 256;
            if (const char* e = tuned ? std::getenv("DOCC_ROCM_GEMV_SLICES") : nullptr) {   // tuning: a cap on the slices
                const int64_t cap = std::atoi(e);
                if (cap >= 1 && cap < slices) slices = cap;
            }
            if (slices < 1 || col_blocks > 0x7fffffffLL) return 1;
            const int64_t chunk = (k + slices - 1) / slices;
            slices = (k + chunk - 1) / chunk;
            // five to eight vectors go as two passes of at most four: two reads of the matrix beat one with eight sums a lane
            char kname[64], fname[64];
            std::snprintf(fname, sizeof(fname), "docc_gemv_colfm_f%d", (int) sizeof(S) * 8);
            PartialsLease partials;
            if (int rcp = partials_for(s, &partials)) return rcp;
            for (int64_t v0 = 0; v0 < nv; v0 += 4) {
                const int64_t gv = nv - v0 < 4 ? nv - v0 : 4;
                std::snprintf(kname, sizeof(kname), "docc_gemv_colpm_%s_v%d_n%d", sizeof(T) == 4 ? "f32" : "f64", lanes, gv <= 2 ? 2 : 4);
                int rcm = launch(kname, (uint32_t) col_blocks, (uint32_t) slices, 1, 256, 0, s, partials.ptr, mat, (long) ldm, vecs + v0 * sx_v,
                                 (long) sx_v, (long) sx_p, (int) gv, (long) k, (long) cols, (long) chunk);
                if (rcm) return rcm;
                const int64_t entries = gv * cols;
                rcm = launch(fname, (uint32_t) ((entries + 63) / 64), 1, 1, 256, 0, s, (const void*) partials.ptr, C + v0 * sy_vec, (long) sy_vec,
                             (long) sy_col, (long) cols, (long) entries, (int) slices, alpha, beta);
                if (rcm) return rcm;
            }
            return 0;
        }
        if (ta || !tb) return 1;
        const bool small_a = m <= n;                  // the vectors: A's rows (m of them) or B's rows (n of them)
        const int64_t nv = small_a ? m : n, big = small_a ? n : m;
        // five to eight vectors: fp64 is faster through the MFMA tiles (8 x 8192 x 8192: 166 us against 218 here), bf16 too
        // once the matrix is large (8 x 28672 x 8192: 111 us against 137; 8 x 8192 x 8192: 56 against 46 here)
        const int64_t max_nv = sizeof(T) == 8 || (sizeof(T) == 2 && big * k > (int64_t(1) << 27)) ? 4 : 8;
        const int vecw = 16 / (int) sizeof(T);
        const bool aligned = ((uintptr_t) (small_a ? B : A) | (uintptr_t) (small_a ? A : B)) % 16 == 0 && (small_a ? ldb : lda) % vecw == 0 &&
                             (small_a ? lda : ldb) % vecw == 0;
        // a wavefront takes four matrix rows, or eight where that still leaves a work-group per CU (fp32 4 x 8192 x 8192:
        // 79 -> 68 us; bf16 gains nothing from it)
        const bool eight = nv <= 4 && aligned && sizeof(T) != 2 && big >= 32 * (int64_t) cus;
        const int64_t wg_rows = eight ? 32 : 16;
        if (nv > max_nv || big < 16 * (int64_t) cus || (big + wg_rows - 1) / wg_rows > 0x7fffffffLL) return 1;
        const T* mat = small_a ? B : A;
        const T* vecs = small_a ? A : B;
        const int64_t ldm = small_a ? ldb : lda, ldx = small_a ? lda : ldb;
        const int64_t sy_row = small_a ? 1 : ldc, sy_vec = small_a ? ldc : 1;
        char kname[64];
        std::snprintf(kname, sizeof(kname), "docc_gemv_rowsm_%s_v%d_n%d%s", sizeof(T) == 2 ? "bf16" : sizeof(T) == 4 ? "f32" : "f64",
                      aligned ? vecw : 1, nv <= 2 ? 2 : nv <= 4 ? 4 : 8, eight ? "_r8" : "");
        return launch(kname, (uint32_t) ((big + wg_rows - 1) / wg_rows), 1, 1, 256, 0, s, mat, (long) ldm, vecs, (long) ldx, (int) nv, C, (long) sy_row,
                      (long) sy_vec, (long) big, (long) k, alpha, beta);
    }
    if (n == 1) {          // y = op(A) b: A as stored is [m][k] (rows form) or [k][m] (columns form)
        M = A, ld = lda, x = B, incx = tb ? 1 : ldb, incy = ldc;
        by_rows = !ta;
        rows = ta ? k : m, cols = ta ? m : k;
    } else if (m == 1) {   // y = a op(B): B as stored is [n][k] (rows form) or [k][n] (columns form)
        M = B, ld = ldb, x = A, incx = ta ? lda : 1, incy = 1;
        by_rows = tb;
        rows = tb ? n : k, cols = tb ? k : n;
    } else {
        return 1;
    }
    const int vec = 16 / (int) sizeof(T);
    const char* type = sizeof(T) == 2 ? "bf16" : sizeof(T) == 4 ? "f32" : "f64";   // elements of the matrix
    const int bits = (int) sizeof(S) * 8;                                        // of the sums and of y
    char name[64];
    if (by_rows) {
        // one wavefront per row: worth it from a few rows per SIMD on
        if (rows < 4 * (int64_t) cus) return 1;
        if ((rows + 3) / 4 > 0x7fffffffLL) return 1;
        const bool aligned = incx == 1 && ((uintptr_t) M | (uintptr_t) x) % 16 == 0 && ld % vec == 0;
        std::snprintf(name, sizeof(name), "docc_gemv_rows_%s_v%d", type, aligned ? vec : 1);
        return launch(name, (uint32_t) ((rows + 3) / 4), 1, 1, 256, 0, s, M, (long) ld, x, (long) incx, C, (long) incy, (long) rows,
                      (long) cols, alpha, beta);
    }
    // columns form: lanes own columns, the rows are sliced so that 2.6 work-groups per CU share the matrix (measured
    // on eight shapes from 4096 x 4096 to 28672 x 8192 against 1.5, 2, 3, 4, 6 and 8 per CU: the fastest on every one,
    // 8192 x 8192 fp32 in 42 us against 50 with eight - fewer slices also leave less for the second launch to add);
    // the slices' sums meet in the stream's partial-results buffer
    if (cols < 256 || rows < 64) return 1;
    const bool aligned = (uintptr_t) M % 16 == 0 && ld % vec == 0 && cols % vec == 0;
    const int lanes = aligned ? vec : 1;
    const int64_t col_blocks = (cols / lanes + 255) / 256;
    int64_t slices = (21 * (int64_t) cus / 8 + col_blocks - 1) / col_blocks;
    if (slices > rows / 16) slices = rows / 16;
    const int64_t fit = (int64_t) kPartialsBytes / ((int64_t) sizeof(S) * cols);
    if (slices > fit) slices = fit;
    if (slices > 256) slices = 256;
    if (const char* e = tuned ? std::getenv("DOCC_ROCM_GEMV_SLICES") : nullptr) {   // tuning: a cap on the slices
        const int64_t cap = std::atoi(e);
        if (cap >= 1 && cap < slices) slices = cap;
    }
    if (slices < 1) return 1;
    const int64_t chunk = (rows + slices - 1) / slices;
    slices = (rows + chunk - 1) / chunk;
    if (col_blocks > 0x7fffffffLL || slices > 65535) return 1;
    PartialsLease partials;
    if (int rcp = partials_for(s, &partials)) return rcp;
    std::snprintf(name, sizeof(name), "docc_gemv_colp_%s_v%d", type, lanes);
    int rc = launch(name, (uint32_t) col_blocks, (uint32_t) slices, 1, 256, 0, s, partials.ptr, M, (long) ld, x, (long) incx, (long) rows,
                    (long) cols, (long) chunk);
    if (rc) return rc;
    std::snprintf(name, sizeof(name), "docc_gemv_colf_f%d", bits);
    return launch(name, (uint32_t) ((cols + 15) / 16), 1, 1, 256, 0, s, (const void*) partials.ptr, C, (long) incy, (long) cols, (int) slices,
                  alpha, beta);
}

// T: element type of A and B; S: type of C, alpha and beta. k_total > 0: the `batch` entries are the parts of a product of that k,
// `k` each and the last one what is left.
template <typename T, typename S = T>
int gemm_launch(const char* prefix, docc_rocm_stream_t stream, int trans_a, int trans_b, int64_t m, int64_t n,
                int64_t k, S alpha, const T* A, int64_t lda, const T* B, int64_t ldb, S beta, S* C, int64_t ldc,
                Picker pick, const S* bias = nullptr,
                int activation = -1, int64_t batch = 1, int64_t batch_a = 0, int64_t batch_b = 0, int64_t batch_c = 0,
                const LinearFinish* fin = nullptr, int64_t k_total = 0) {
    if ((trans_a != DOCC_ROCM_NO_TRANS && trans_a != DOCC_ROCM_TRANS) ||
        (trans_b != DOCC_ROCM_NO_TRANS && trans_b != DOCC_ROCM_TRANS))
        return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "%s: transpose code must be 111 or 112", prefix);
    if (m < 0 || n < 0 || k < 0) return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "%s: negative dimension", prefix);
    const bool ta = trans_a == DOCC_ROCM_TRANS, tb = trans_b == DOCC_ROCM_TRANS;
    const int64_t a_cols = ta ? m : k, b_cols = tb ? k : n;
    if (lda < (a_cols > 1 ? a_cols : 1) || ldb < (b_cols > 1 ? b_cols : 1) || ldc < (n > 1 ? n : 1))
        return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "%s: leading dimension too small (lda=%lld ldb=%lld ldc=%lld)",
                    prefix, (long long) lda, (long long) ldb, (long long) ldc);
    if (activation < -1 || activation > DOCC_ROCM_UNARY_ERF)
        return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "%s: unknown activation %d", prefix, activation);
    if (activation >= 0 && activation != DOCC_ROCM_UNARY_RELU && activation != DOCC_ROCM_UNARY_ABS)
        return fail(DOCC_ROCM_ERR_UNSUPPORTED, "%s: only ReLU and Abs are built into the GEMM store (activation %d)", prefix, activation);
    if (batch < 0 || batch > 65535) return fail(DOCC_ROCM_ERR_UNSUPPORTED, "%s: batch must be 0..65535", prefix);
    if (batch_a < 0 || batch_b < 0 || batch_c < 0) return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "%s: negative batch stride", prefix);
    if (m == 0 || n == 0 || batch == 0) return 0;
    if (batch > 1 && batch_c < (m - 1) * ldc + n) return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "%s: the C matrices of the batch overlap", prefix);
    if ((!C && !fin) || (k > 0 && (!A || !B))) return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "%s: null pointer", prefix);
    int rc = ensure_device();
    if (rc) return rc;
    hipStream_t s = (hipStream_t) stream;
    char name[96];
    const bool tuned = gemm_tuning_set();
    const int cus = cu_count();
    auto tuning = [&](const char* variable) -> const char* { return tuned ? std::getenv(variable) : nullptr; };
    // A block of the device block cache for this call, given back behind its last launch. False: there is none (no memory, or a
    // capture it could not be kept for), and the product runs in a form without it.
    auto block = [&](void** ptr, int64_t bytes) { return !foreign_capture(s) && docc_rocm_malloc_async(ptr, (size_t) bytes, stream) == 0; };
    // with a finish (docc_rocm_linear): where no kernel has it in its store, the product goes to a block of the device block
    // cache and the chain runs as one pass over it. `product(C)` returns 1 where it does not take the shape.
    auto through_memory = [&](auto&& product) -> int {
        if (foreign_capture(s))
            return fail(DOCC_ROCM_ERR_UNSUPPORTED, "linear: this shape needs device memory between its launches, which a capture that the runtime did not begin cannot keep");
        void* wide = nullptr;
        if (int r = docc_rocm_malloc_async(&wide, (size_t) (m * n) * sizeof(S), stream)) return r;
        int r = product((S*) wide);
        if (r == 0) r = finish_parts(s, wide, m, n, 1, 1.0f, *fin);
        const int r2 = docc_rocm_free_async(wide, stream);
        return r ? r : r2;
    };
    auto plain_product = [&](S* to) {
        return gemm_launch<T, S>(prefix, stream, trans_a, trans_b, m, n, k, alpha, A, lda, B, ldb, (S) 0, to, n, pick);
    };
    if (fin && (k == 0 || alpha == (S) 0)) return through_memory(plain_product);
    if (k == 0 || alpha == (S) 0) {   // an empty product, or one BLAS does not reference ("when ALPHA is zero ...")
        std::snprintf(name, sizeof(name), "docc_%s_scale_c", prefix);
        int64_t blocks = (m * n + 255) / 256;
        if (blocks > 4096) blocks = 4096;
        for (int64_t z = 0; z < batch && rc == 0; z++)   // an empty product: one small launch per entry
            rc = launch(name, (uint32_t) blocks, 1, 1, 256, 0, s, C + z * batch_c, (long) m, (long) n, (long) ldc, beta);
        if (rc || (!bias && activation < 0)) return rc;
        if (batch > 1) return fail(DOCC_ROCM_ERR_UNSUPPORTED, "%s: k == 0 or alpha == 0 with an epilogue and a batch", prefix);
        // the epilogue of an empty product: C = act(beta * C + bias), through the elementwise kernel
        if (ldc != n) return fail(DOCC_ROCM_ERR_UNSUPPORTED, "%s: k == 0 or alpha == 0 with an epilogue needs ldc == n", prefix);
        const int64_t shape[2] = {m, n}, row[2] = {1, n};
        const int post[1] = {activation};
        return docc_rocm_elementwise_fused(stream, sizeof(S) == 8 ? 64 : 32, 2, shape, bias ? DOCC_ROCM_BINARY_ADD : -1, shape, C, 0.0,
                                           bias ? row : nullptr, bias, 0.0, activation >= 0 ? 1 : 0, post, C);
    }
    // A layer whose product has too few tiles for the kernels below to fill the compute units, weights stored [n][k]: K cut between the wavefronts of a work-group,
    // the chain in the same launch (csrc/kernels/gemm_waves.hip). DOCC_ROCM_GEMM_WAVES=0 switches it off, =16, =32, =64 and =1 take the tile of that size, or that
    // of a work-group a compute unit (tests, tuning).
    if constexpr (sizeof(T) <= 4) {
        const char* waves_env = tuning("DOCC_ROCM_GEMM_WAVES");
        int forced = waves_env ? std::atoi(waves_env) : -1;
        for (const char* other : {"DOCC_ROCM_GEMM_CFG", "DOCC_ROCM_GEMM_TILE", "DOCC_ROCM_GEMM_SPLITK", "DOCC_ROCM_GEMM_SKINNY"})   // they ask for another form
            if (forced < 0 && tuning(other)) forced = 0;
        if (fin && !ta && tb && batch == 1 && forced != 0 && n % 8 == 0 && waves_shape_ok(m, n, k, lda, ldb, true, sizeof(T)) &&
            ((uintptr_t) A | (uintptr_t) B | (uintptr_t) fin->bias | (uintptr_t) fin->residual | (uintptr_t) fin->out) % 16 == 0) {
            const bool on_lines = ((uintptr_t) A | (uintptr_t) B | (uintptr_t) (lda * (int64_t) sizeof(T)) | (uintptr_t) (ldb * (int64_t) sizeof(T))) % 128 == 0;
            const WavesChoice w = waves_choice(m, n, k, cus, sizeof(T), on_lines, forced);
            // Up to 32 rows (against the kernels with K in parts and a pass behind them): bf16 1 x 2048 -> 8192 9.9 us and 7.8, 8 x 2048 -> 8192 12.7 and 7.8,
            // 16 x 12288 -> 3072 21.3 and 14.2, 32 x 4096 -> 1024 14.6 and 5.6; fp32 21.2 and 12.7 (8 x 2048), 40.6 and 35.3, 16.2 and 9.1. But a single row of
            // a large matrix is read by the matrix-vector kernel: fp32 1 x 4096 -> 14336 42.6 us here and 39.7, bf16 1 x 8192 -> 28672 78.8 and 73.4; a block of 1 x 3072
            // whose weights come from HBM 66.6 us and 59.0, in bf16 38.0 and 36.2.
            // Beyond by the estimates: bf16 1024 x 1024 x 256 9.9 -> 5.8 us, 1024 x 256 x 1024 13.8 -> 5.3, 1024 x 512 x 2048 14.2 -> 8.2, 512 x 4096 x 1024 15.0 ->
            // 11.7, but 1024 x 4096 x 1024 17.3 and 20.7; fp32 1024 x 256 x 1024 13.1 -> 8.6, 256 x 2048 x 512 13.5 -> 8.6, 2048 x 3072 x 768 108 -> 86, but
            // 2048 x 2048 x 512 41.5 and 43.6. (Both estimates are some 10 % off: for a clear gain only.)
            const bool few = m <= 32 && (m > 1 || n * k * (int64_t) sizeof(T) < (int64_t(64) << 20));
            if (forced > 0 || few || (m > 32 && w.seconds < 0.85 * tiles_seconds(pick, m, n, k, true, cus, sizeof(T), on_lines))) {
                const int64_t tiles = ((m + w.edge - 1) / w.edge) * ((n + w.edge - 1) / w.edge);
                std::snprintf(name, sizeof(name), "docc_%cgemm_waves_%dx%d%s_f", sizeof(T) == 2 ? 'b' : 's', w.edge, w.edge, w.one ? "_one" : "");
                // a ring of two pieces of 16 bytes times `seg` of the tile's rows and columns a wavefront; the sums of all of them, or of half, take less
                const int nw = w.edge == 16 || (w.one && sizeof(T) == 4) ? 8 : 4, seg = w.edge <= 32 || (w.one && sizeof(T) == 2) ? 8 : 4;
                return launch(name, (uint32_t) tiles, 1, 1, 64 * nw, (uint32_t) (nw * 2 * 2 * w.edge * seg * 16), s, A, (long) lda, B, (long) ldb, (long) m, (long) n, (long) k,
                              (float) alpha, *fin);
            }
        }
    }
    auto waves_plain = [&](const WavesChoice& w) {
        const int64_t tiles = ((m + w.edge - 1) / w.edge) * ((n + w.edge - 1) / w.edge);
        std::snprintf(name, sizeof(name), "docc_%cgemm_waves_%dx%d%s_n%c", prefix[0], w.edge, w.edge, w.one ? "_one" : "", tb ? 't' : 'n');
        // the rings, or the sums of all wavefronts or (above 64 KB) of half of them
        const int64_t nw = w.edge == 16 || (w.one && sizeof(T) > 2) ? 8 : 4, seg = w.edge <= 32 || (w.one && sizeof(T) == 2) ? 8 : 4;
        const int64_t ring = nw * 2 * 2 * w.edge * seg * 16, sums = nw * w.edge * (w.edge * (int64_t) sizeof(S) + 16), held = sums > 65536 ? sums / 2 : sums;
        return launch(name, (uint32_t) tiles, 1, 1, (uint32_t) (64 * nw), (uint32_t) (ring > held ? ring : held), s, A, (long) lda, B, (long) ldb, (long) m, (long) n, (long) k, alpha, beta, C,
                      (long) ldc, bias, activation);
    };
    // The same for a product of fp32 or fp64 alone, B stored [k][n] as well (csrc/kernels/gemm_waves_plain.hip).
    if (sizeof(T) > 2 && !fin && !ta && batch == 1 && (activation < 0 || activation == DOCC_ROCM_UNARY_ABS || activation == DOCC_ROCM_UNARY_RELU) && n >= 16 && waves_shape_ok(m, n, k, lda, ldb, tb, sizeof(T)) && ((uintptr_t) A | (uintptr_t) B) % 16 == 0) {
        const char* waves_env = tuning("DOCC_ROCM_GEMM_WAVES");
        int forced = waves_env ? std::atoi(waves_env) : -1;
        for (const char* other : {"DOCC_ROCM_GEMM_CFG", "DOCC_ROCM_GEMM_TILE", "DOCC_ROCM_GEMM_SPLITK", "DOCC_ROCM_GEMM_SKINNY", "DOCC_ROCM_GEMV_OFF", "DOCC_ROCM_GEMV_SLICES"})
            if (forced < 0 && tuning(other)) forced = 0;
        bool pays = false;
        const bool on_lines = ((uintptr_t) A | (uintptr_t) B | (uintptr_t) (lda * (int64_t) sizeof(T)) | (uintptr_t) (ldb * (int64_t) sizeof(T))) % 128 == 0;
        const WavesChoice w = waves_choice(m, n, k, cus, sizeof(T), on_lines || !tb, forced);
        if (m > 32) {
            // by the estimates: fp32 512 x 512 x 512 10.6 -> 6.2 us, 192 x 64 x 1664 11.6 -> 5.6, 64 x 5824 x 896 15.7 -> 12.7;
            // fp64 512 x 512 x 512 12.0 -> 8.6
            // (315 x 600 x 3584, B [k][n] 23.2 us and 26.2: not above k = 2048 there). Of 700 drawn products with B [n][k], k a multiple of 128 or not, 412 changed, fp32 1.47
            // times as fast and fp64 1.34 (geometric means; 7 % slower at most); below 64 and 128 k a launch of either takes 5 us (52 x 1512 x 32 in fp64 4.5 and 6.0). From 40 us on the other estimate is
            // too high by a quarter in fp64: 1242 x 251 x 3584 59 us for 47, on tiles of 16 x 16 here 51 (those of 32 x 32 still win there: 216 x 906 x 3844 44.3 -> 39.7).
            const double margin = sizeof(T) == 8 && w.edge == 16 && w.seconds > 40e-6 ? 0.7 : 0.85;
            pays = forced < 0 && (tb ? k >= (sizeof(T) == 4 ? 64 : 128) : k <= 2048) && w.seconds < margin * tiles_seconds(pick, m, n, k, tb, cus, sizeof(T), on_lines);
        } else if (tb) {
            // Against the matrix-vector kernels, the skinny ones and K in parts, B stored [n][k]: fp32 2 x 8192 x 2048 24 -> 12 us, 8 x 2048 x 2048 11.2 -> 6.1, 32 x
            // 8192 x 8192 96 -> 59; fp64 8 x 8192 x 2048 40 -> 22, but 8 x 512 x 8192 19.5 and 23.4
            // (few tiles, a long chain each). From two tiles on. A single row is one launch there too (fp32 1 x 2048 x 8192 11.7 us, 13.9 here), but for few columns.
            pays = n >= 32 && n * k <= (int64_t(1) << 27) && (m > 1 || n < 4 * (int64_t) cus) && (sizeof(T) != 8 || k <= 4096 || (m > 1 && n >= 2048));
        } else {
            // B stored [k][n]: fp32 1 x 2048 x 2048 9.4 -> 6.6 us, 8 x 8192 x 512 11.2 -> 5.6, but 2 x 8192 x 8192 46.6 and 69 (64 bytes of a row of B a work-group);
            // fp64 8 x 2048 x 2048 15.3 -> 9.6
            pays = k <= 2048 && n * k <= (int64_t(1) << 24);
        }
        if (forced > 0 || (pays && forced < 0)) return waves_plain(w);
    }
    const bool epilogue = bias || activation >= 0;
    // A tall matrix times a few columns held as numpy holds them (B [k][n], n small): rows of B are a few elements long, so
    // the kernels that read whole vectors along n do not apply (n = 2, 5, 9 ... went through the element-wise tiles at a
    // ninth of the rate) and the matrix-vector kernels want the vectors contiguous along k. B is small: it is transposed
    // into a block of the device block cache first (k x n elements), and the product runs as A B'^T.
    if (!tb && batch == 1 && n >= 2 && n <= 64 && ldb == n && m >= 1024 && k >= 256 && k % (16 / (int64_t) sizeof(T)) == 0 &&
        (n <= 4 || n % (16 / (int64_t) sizeof(T)) != 0) && !tuning("DOCC_ROCM_GEMV_OFF")) {
        if (fin) return through_memory(plain_product);
        void* bt = nullptr;
        if (block(&bt, n * k * (int64_t) sizeof(T))) {
            const int64_t shape[2] = {k, n}, perm[2] = {1, 0};
            rc = docc_rocm_transpose(stream, (int) sizeof(T), 2, shape, perm, B, bt);
            if (!rc)
                rc = gemm_launch<T, S>(prefix, stream, trans_a, DOCC_ROCM_TRANS, m, n, k, alpha, A, lda, (const T*) bt, k, beta, C, ldc, pick, bias, activation);
            const int rc2 = docc_rocm_free_async(bt, stream);
            return rc ? rc : rc2;
        }
    }
    // Five to 32 rows of fp32 against a wide matrix go to the kernels of csrc/kernels/gemm_skinny.hip (below); measured against
    // the tiles with K in parts and the matrix-vector forms, they pay from 8 M elements of B (16 M above 16 rows).
    // DOCC_ROCM_GEMM_SKINNY=1 takes them for smaller ones too (tests).
    const char* skinny_env = tuning("DOCC_ROCM_GEMM_SKINNY");
    const bool skinny_on = !(skinny_env && skinny_env[0] == '0'), skinny_any_size = skinny_env && skinny_env[0] == '1';
    // (a lane's offset from the chunk's base, up to 31 rows of either operand, is held in 32 bits)
    const bool skinny_base = batch == 1 && !ta && (!epilogue || ldc == n) && n >= 512 && k >= 512 && skinny_on && (uintptr_t) A % 16 == 0 &&
                             (uintptr_t) B % 16 == 0 && lda < (int64_t(1) << 26) && ldb < (int64_t(1) << 26);
    // (B stored [n][k]: from 3 rows, where the matrix-vector form for several vectors falls behind - 4 x 8192 x 8192 67 -> 57 us,
    // 4 x 4096 x 11008 62 -> 48 - but up to 8 rows not above 128 M elements, where that form is the faster one again)
    const bool skinny_f32 = sizeof(T) == 4 && skinny_base && m >= (skinny_any_size ? 2 : tb ? 3 : 5) && m <= (tb ? 16 : 32) &&
                            !(tb && m <= 8 && n * k > (int64_t(1) << 27)) &&
                            (n * k >= (m <= 16 ? int64_t(8) << 20 : int64_t(16) << 20) || skinny_any_size) && lda % 4 == 0 && ldb % 4 == 0 &&
                            k % 4 == 0 && (tb || n % 4 == 0);
    // bf16 with B stored [n][k] (a layer's weights): 3 to 32 rows (two rows are faster as matrix-vector products, 64 on the tiles)
    const bool skinny_bf16 = sizeof(T) == 2 && skinny_base && tb && m >= 3 && m <= 32 && (n * k >= (int64_t(8) << 20) || skinny_any_size) &&
                             lda % 8 == 0 && ldb % 8 == 0 && k % 8 == 0;
    // fp64 with B stored [k][n]: 5 to 16 rows (up to four are matrix-vector products, above 16 the tiles)
    const bool skinny_f64 = sizeof(T) == 8 && skinny_base && !tb && m >= 5 && m <= 16 && (n * k >= (int64_t(4) << 20) || skinny_any_size) &&
                            lda % 2 == 0 && ldb % 2 == 0 && k % 2 == 0 && n % 2 == 0;
    const bool skinny = skinny_f32 || skinny_bf16 || skinny_f64;
    if (fin && (m <= 8 || n <= 8) && !skinny && batch == 1 && !foreign_capture(s)) {
        rc = through_memory([&](S* to) { return gemv_launch<T, S>(prefix, s, ta, tb, m, n, k, alpha, A, lda, B, ldb, (S) 0, to, n, tuned, cus); });
        if (rc != 1) return rc;
    } else if (!fin && (m <= 8 || n <= 8) && !skinny && batch == 1 && (!epilogue || ldc == n)) {
        rc = gemv_launch<T, S>(prefix, s, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, tuned, cus);
        if (rc == 0 && epilogue) {
            // the few rows or columns of output are a small tensor: bias and activation as one elementwise pass over it,
            // the same roundings as the fused store
            const int64_t shape[2] = {m, n}, row[2] = {1, n};
            const int post[1] = {activation};
            return docc_rocm_elementwise_fused(stream, sizeof(S) == 8 ? 64 : 32, 2, shape, bias ? DOCC_ROCM_BINARY_ADD : -1, shape, C, 0.0,
                                               bias ? row : nullptr, bias, 0.0, activation >= 0 ? 1 : 0, post, C);
        }
        if (rc != 1) return rc;
    }
    const size_t vec = 16 / sizeof(T);
    // the aligned kernels read whole 128-bit vectors: pointers, leading dimensions and the
    // contiguous extents of both operands must be multiples of the vector length
    const int64_t a_contig = ta ? m : k, b_contig = tb ? k : n;
    const bool vectors = ((uintptr_t) A % 16 == 0) && ((uintptr_t) B % 16 == 0) && (lda % vec == 0) && (ldb % vec == 0) &&
                         (a_contig % (int64_t) vec == 0) && (b_contig % (int64_t) vec == 0) &&
                         (batch == 1 || (batch_a % (int64_t) vec == 0 && batch_b % (int64_t) vec == 0));
    const bool lines = vectors && ((uintptr_t) A | (uintptr_t) B | (uintptr_t) (lda * (int64_t) sizeof(T)) | (uintptr_t) (ldb * (int64_t) sizeof(T))) % 128 == 0;
    const int aligned = lines ? 2 : vectors ? 1 : 0;
    // A few rows against a wide fp32 matrix: B goes from global memory straight into the MFMA operands, 128 columns of one part
    // of K per work-group, the parts added in order by a second launch. With B stored [n][k] the lanes of a load walk different
    // rows, which pays up to 16 rows only. DOCC_ROCM_GEMM_SKINNY=0 switches it off, DOCC_ROCM_GEMM_SPLITK forces the number of
    // parts (tests, tuning).
    if (skinny) {
        {
            // fp32: 16 or 32 rows per MFMA, 128 columns per work-group; bf16: 1, 2 or 4 blocks of 16 rows, 64 columns
            const int nw = 4, nbuf = 2;
            const int ch = skinny_bf16 ? 64 : tb ? 32 : 16, mt = skinny_bf16 ? (m <= 16 ? 1 : 2) : m <= 16 ? 16 : 32;
            const int64_t col_blocks = skinny_bf16 || skinny_f64 ? (n + 63) / 64 : (n + 127) / 128;
            const int64_t unit = (int64_t) nw * ch;
            auto part_length = [&](int64_t parts) { return ((k + parts - 1) / parts + unit - 1) / unit * unit; };
            // The number of parts: measured on 4096 x 4096, 8192 x 8192, 11008 x 4096 and 4096 x 11008, what counts is that
            // the work-groups come out as whole rounds over the CUs (8192 x 8192: 4, 8 and 12 parts 48-51 us, 6 parts 56 us),
            // then few parts (their products are written and read again) and 128 and more k per wavefront.
            int64_t parts = 1;
            double best = -1.0;
            for (int64_t p = 1; p <= 64 && part_length(p) >= nw * 64 && p * 16 * m <= k; p++) {
                const int64_t kp = part_length(p);
                if ((k + kp - 1) / kp != p) continue;   // rounding to whole chunks made it fewer parts
                // B stored [n][k]: a lane walks its row of B, and parts longer than 4096 ran a quarter slower (bf16 16384 x 16384
                // in 1 or 2 parts 127 us, in 4 parts 97)
                if (tb && kp > 4096 && part_length(p + 1) >= nw * 64) continue;
                const double per_cu = (double) (col_blocks * p) / cus;
                const double score = per_cu / (double) (int64_t) (per_cu + 0.999999) - 0.01 * (double) p - (kp < nw * 128 ? 0.15 : 0.0);
                if (score > best) {
                    best = score;
                    parts = p;
                }
            }
            if (const char* e = tuning("DOCC_ROCM_GEMM_SPLITK"))
                if (std::atoll(e) > 0 && part_length(std::atoll(e)) >= unit) parts = std::atoll(e);
            const int64_t kpart = part_length(parts);
            parts = (k + kpart - 1) / kpart;
            const int64_t bytes = parts * m * n * (int64_t) sizeof(S);
            const bool direct = !fin && parts == 1 && (tb || ((uintptr_t) C % 16 == 0 && ldc % (skinny_f64 ? 2 : 4) == 0));
            const bool own_block = !direct && bytes > (int64_t) kPartialsBytes;
            void* buf = nullptr;
            if (direct || (bytes <= (int64_t(64) << 20) && (!own_block || block(&buf, bytes)))) {
                PartialsLease lease;
                if (!direct && !own_block) {
                    if ((rc = partials_for(s, &lease))) return rc;
                    buf = lease.ptr;
                }
                if (skinny_f64)
                    std::snprintf(name, sizeof(name), "docc_dgemm_skinny16_nn_w%d_b%d", nw, nbuf);
                else if (skinny_bf16)
                    std::snprintf(name, sizeof(name), "docc_bgemm_skinny%d_nt_w%d_b%d", mt, nw, nbuf);
                else
                    std::snprintf(name, sizeof(name), "docc_sgemm_skinny%d_n%c_w%d_c%d_b%d", mt, tb ? 't' : 'n', nw, ch, nbuf);
                const uint32_t slot_bytes = skinny_bf16 ? 4096u * mt : mt == 32 && !skinny_f64 ? 16384u : 8192u;   // a wavefront's block of sums
                rc = launch(name, (uint32_t) col_blocks, (uint32_t) parts, 1, 64 * nw, (uint32_t) (nw / 2) * slot_bytes, s, A, (long) lda, B, (long) ldb,
                            direct ? (void*) C : buf, (long) (direct ? ldc : n), (long) m, (long) n, (long) k, (long) kpart, alpha, beta,
                            direct ? 1 : 0);
                if (!rc && fin) {
                    rc = finish_parts(s, buf, m, n, (int) parts, (float) alpha, *fin);
                } else if (!rc && !direct) {
                    int64_t blocks = (m * n + 255) / 256;
                    if (blocks > 4096) blocks = 4096;
                    rc = launch(sizeof(S) == 8 ? "docc_splitk_combine_f64" : "docc_splitk_combine_f32", (uint32_t) blocks, 1, 1, 256, 0, s, (const S*) buf, C,
                                (long) m, (long) n, (long) ldc, (int) parts, alpha, beta);
                }
                if (own_block) {
                    const int rc2 = docc_rocm_free_async(buf, stream);
                    if (!rc) rc = rc2;
                }
                if (rc || !epilogue) return rc;
                // the few rows of output are a small tensor: bias and activation as one elementwise pass over it, the same
                // roundings as the fused store
                const int64_t shape[2] = {m, n}, row[2] = {1, n};
                const int post[1] = {activation};
                return docc_rocm_elementwise_fused(stream, sizeof(S) == 8 ? 64 : 32, 2, shape, bias ? DOCC_ROCM_BINARY_ADD : -1, shape, C, 0.0,
                                                   bias ? row : nullptr, bias, 0.0, activation >= 0 ? 1 : 0, post, C);
            }
        }
    }
    // Operands the vectors of the asynchronous kernels do not fit are packed first (csrc/kernels/gemm_pack.hip): those that are
    // off, both of them where k itself is no whole number of vectors. That costs a launch of 4-5 us and reading and writing the operands
    // once; the element-wise tiles sustain a tenth (bf16 read along m or n) to nine tenths (fp64) of the others' rate, and wait for every
    // step of a long k. Measured, k one off the vector: bf16 4096^3 649-1195 us plain against 134-208 packed, 512^3 13-27 against 12;
    // fp32 2048^3 190-310 against 148-272, 2800 x 517 x 3565 194 against 139, but 5120 x 2304 x 1391 312 against 359 (360 tiles: two
    // rounds); fp64 6537 x 5561 x 221 289 against 329, 915 x 1581 x 3707 272 against 204. fp32 and fp64 weigh both forms in rounds over the CUs: of 220
    // drawn products 6 are more than 5 % slower than plain (33 by the rates alone), in the mean 0.8 % off the better form (2.7 %).
    // DOCC_ROCM_GEMM_PACK=0 switches it off, =1 packs whatever the size (tests, tuning).
    const char* pack_env = tuning("DOCC_ROCM_GEMM_PACK");
    if (!aligned && batch == 1 && !(pack_env && pack_env[0] == '0')) {
        const int64_t v = (int64_t) vec;
        const bool whole_k = k % v == 0;
        auto off = [&](const T* p, int64_t ld, int64_t contiguous) { return (uintptr_t) p % 16 != 0 || ld % v != 0 || contiguous % v != 0; };
        const bool pack_a = !whole_k || off(A, lda, a_contig), pack_b = !whole_k || off(B, ldb, b_contig);
        const bool turned = (pack_a && ta) || (pack_b && !tb);   // an operand would be read along m or n
        const double work = (double) m * (double) n * (double) k;
        const int64_t kp = pack_a && pack_b ? (k + 63) / 64 * 64 : k;
        const int64_t bytes_a = pack_a ? m * kp * (int64_t) sizeof(T) : 0, bytes_b = pack_b ? n * kp * (int64_t) sizeof(T) : 0;
        bool pays = false;
        if (sizeof(T) == 2) {
            // the plain tiles: the chain of K-steps of one tile, or all of them at the rate they sustain; against the copies and the rate of
            // the asynchronous ones (flop per us)
            const double chain_us = (turned ? 2.3 : 0.95) * (double) k / 64, all_us = 2.0 * work / (turned ? 1.2e8 : 4.2e8);
            // (below k = 192 both are bound by storing C)
            pays = (chain_us > 14.0 || k >= 192) &&
                   5.0 + (chain_us > all_us ? chain_us : all_us) > 14.0 + 2e-6 / 4.0 * (double) (bytes_a + bytes_b) + 2.0 * work / 1.1e9;
        } else {
            pays = k >= 192 && plain_us(pick, m, n, k, tb, turned, cus, sizeof(T)) >
                                   8.0 + 0.9e-7 * (double) (bytes_a + bytes_b) + 1e6 * sdgemm_best_seconds(pick, m, n, kp, pack_b || tb, cus, sizeof(T));
        }
        if (pack_env && pack_env[0] == '1') pays = true;
        const int64_t tiles_k = (kp + 63) / 64;
        const int64_t groups_a = pack_a ? (m + 63) / 64 * tiles_k : 0, groups_b = pack_b ? (n + 63) / 64 * tiles_k : 0;
        const int64_t at_b = (bytes_a + 255) / 256 * 256;
        void* packed = nullptr;
        if (pays && bytes_a + bytes_b <= (int64_t(1) << 31) && groups_a + groups_b < (int64_t(1) << 24) && block(&packed, at_b + bytes_b)) {
            struct {
                const void* src;
                void* dst;
                long ld, rows;
                int k_major;
            } pa{A, packed, (long) lda, (long) m, ta}, pb{B, (char*) packed + at_b, (long) ldb, (long) n, !tb};
            rc = launch(sizeof(T) == 2 ? "docc_gemm_pack_b2" : sizeof(T) == 4 ? "docc_gemm_pack_b4" : "docc_gemm_pack_b8",
                        (uint32_t) (groups_a + groups_b), 1, 1, 256, 0, s, pa, pb, (long) groups_a, (long) k, (long) kp);
            if (!rc)
                rc = gemm_launch<T, S>(prefix, stream, pack_a ? DOCC_ROCM_NO_TRANS : trans_a, pack_b ? DOCC_ROCM_TRANS : trans_b, m, n, kp, alpha,
                                       pack_a ? (const T*) pa.dst : A, pack_a ? kp : lda, pack_b ? (const T*) pb.dst : B, pack_b ? kp : ldb, beta, C, ldc,
                                       pick, bias, activation, 1, 0, 0, 0, fin);
            const int rc2 = docc_rocm_free_async(packed, stream);
            return rc ? rc : rc2;
        }
    }
    // DOCC_ROCM_GEMM_TILE=big|small overrides the size heuristic (tests, tuning)
    const char* force = tuning("DOCC_ROCM_GEMM_TILE");
    TileConfig cfg = pick(m, n, k, tb, batch, aligned, force && force[0] == 'b' ? 1 : force && force[0] == 's' ? -1 : 0, cus);
    // DOCC_ROCM_GEMM_CFG=BMxBNxBKxWAVES[xSTAGES[p|q]] selects a built configuration directly (tuning)
    if (const char* c = tuning("DOCC_ROCM_GEMM_CFG")) {
        TileConfig t{};
        char tag = 0;
        const int got = std::sscanf(c, "%dx%dx%dx%dx%d%c", &t.bm, &t.bn, &t.bk, &t.waves, &t.stages, &tag);
        t.spread = got == 6 && tag == 'p';
        t.small = got == 6 && tag == 'q';
        if (got >= 4 && t.bm > 0 && t.bn > 0 && t.bk > 0 && t.waves > 0) cfg = t;
    }
    // the 16x16x32 kernels (gemm_async16.h) take whole pairs of K-steps, at least a ring of them, in the last part too
    const int64_t k_last = k_total > 0 ? k_total - (batch - 1) * k : k;
    for (int64_t kk : {k, k_last})
        if (cfg.small && !(kk % (2 * cfg.bk) == 0 && kk >= (int64_t) cfg.stages * cfg.bk)) cfg.small = false;
    // the asynchronous kernels need aligned operands and address a tile with 32-bit byte offsets
    const int64_t max_edge = cfg.bm > cfg.bn ? (cfg.bm > cfg.bk ? cfg.bm : cfg.bk) : (cfg.bn > cfg.bk ? cfg.bn : cfg.bk);
    const bool offsets_fit = max_edge * (lda > ldb ? lda : ldb) * (int64_t) sizeof(T) < (int64_t(1) << 32);
    if (cfg.stages > 0 && !(aligned && offsets_fit)) cfg = pick(m, n, k, tb, batch, 0, 0, cus);
    const int64_t tiles = ((m + cfg.bm - 1) / cfg.bm) * ((n + cfg.bn - 1) / cfg.bn);
    if (tiles > 0x7fffffffLL) return fail(DOCC_ROCM_ERR_UNSUPPORTED, "%s: too many tiles", prefix);
    // Few output tiles and a long K extent (a handful of rows against a wide matrix: the product is bound by reading
    // that matrix, and a work-group per tile reads it on a few CUs only): K is cut into parts, each part's product is
    // one entry of a batched launch into the stream's buffer of partial results, and a second launch adds the parts
    // (in order: the result does not depend on the device's scheduling). DOCC_ROCM_GEMM_SPLITK=0 switches it off,
    // another number forces that many parts where K allows it (tests, tuning).
    const bool largest_fits = 256 * (lda > ldb ? lda : ldb) * (int64_t) sizeof(T) < (int64_t(1) << 32);   // whatever tile the parts take
    if (batch == 1 && (!epilogue || ldc == n) && cfg.stages > 0 && largest_fits && k >= 512) {
        const char* env = tuning("DOCC_ROCM_GEMM_SPLITK");
        // the parts' products: in the stream's buffer of partial results where they fit, else in a block of the device
        // block cache (taken and returned in stream order), up to 64 MiB; in a capture that keeps no blocks only in a buffer that is there
        const int64_t max_bytes = !foreign_capture(s) ? kMaxPartsBytes : partials_held(s) ? (int64_t) kPartialsBytes : 0;
        auto part_of = [&](int64_t parts) { return part_length(k, parts); };
        auto allowed = [&](int64_t parts) {
            const int64_t part = part_of(parts);
            return parts <= 64 && (k + part - 1) / part == parts && part >= 256 && parts * m * n * (int64_t) sizeof(S) <= max_bytes;
        };
        // Estimated seconds of the product in `parts` parts on the tile the picker gives that many matrices, plus writing and reading the
        // parts at 5 TB/s and a second launch.
        // (the second launch of a bf16 product counts 3.5 us: with 2 us 25 of 274 drawn products were cut that gained a tenth at most or lost, and a
        // feed-forward block of 3 tokens x 192, which is bound by its launches, took 23.7 us instead of 20.6)
        const double behind = epilogue ? 4e-6 : 0.0;   // bias and activation are a launch of their own then (64 x 192 x 1093 bf16 whole 12 us, in parts 15)
        auto seconds = [&](const TileConfig& c, int64_t parts) {
            if (sizeof(T) == 2)
                return bgemm_seconds(c, m, n, part_of(parts), tb, parts, cus, lines) + (parts > 1 ? 2.0 * (double) parts * (double) m * (double) n * sizeof(S) / 5e12 + 3.5e-6 + behind : 0.0);
            double t = sdgemm_seconds(c, m, n, k, parts, cus, sizeof(T));
            if (parts > 1) t += 2.0 * (double) parts * (double) m * (double) n * sizeof(S) / 5e12 + 3e-6 + behind;
            return t;
        };
        int64_t splits = 1;
        if (env) {
            const int64_t wanted = std::atoll(env);
            while (splits * 2 <= wanted && allowed(splits * 2)) splits *= 2;
        } else if (tiles < cus) {   // CUs without a work-group: the case parts are for
            double best = seconds(cfg, 1);
            for (const int64_t parts : kPartCounts) {
                if (!allowed(parts)) continue;
                const TileConfig c = pick(m, n, part_of(parts), tb, parts, aligned, 0, cus);
                if (c.stages == 0) break;
                const double t = seconds(c, parts);
                if (t < (splits > 1 ? 1.0 : sizeof(T) == 2 ? 0.95 : 0.9) * best) {   // cut for a clear gain only: the estimate is rough
                    best = t;
                    splits = parts;
                }
            }
        }
        const int64_t bytes = splits * m * n * (int64_t) sizeof(S);
        const bool own_block = bytes > (int64_t) kPartialsBytes;
        PartialsLease lease;
        void* parts = nullptr;
        if (splits >= 2 && (own_block ? block(&parts, bytes) : partials_for(s, &lease) == 0)) {
            if (!own_block) parts = lease.ptr;
            const int64_t part = part_of(splits);
            rc = gemm_launch<T, S>(prefix, stream, trans_a, trans_b, m, n, part, (S) 1, A, lda, B, ldb, (S) 0, (S*) parts, n, pick, nullptr, -1, splits,
                                   ta ? part * lda : part, tb ? part : part * ldb, m * n, nullptr, k);
            if (!rc && fin) {
                rc = finish_parts(s, parts, m, n, (int) splits, (float) alpha, *fin);
            } else if (!rc) {
                int64_t blocks = (m * n + 255) / 256;
                if (blocks > 4096) blocks = 4096;
                rc = launch(sizeof(S) == 8 ? "docc_splitk_combine_f64" : "docc_splitk_combine_f32", (uint32_t) blocks, 1, 1, 256, 0, s, (const S*) parts, C,
                            (long) m, (long) n, (long) ldc, (int) splits, alpha, beta);
            }
            if (own_block) {
                const int rc2 = docc_rocm_free_async(parts, stream);
                if (!rc) rc = rc2;
            }
            if (rc || !epilogue) return rc;
            // bias and activation as one elementwise pass over the output, the same roundings as the fused store
            const int64_t shape[2] = {m, n}, row[2] = {1, n};
            const int post[1] = {activation};
            return docc_rocm_elementwise_fused(stream, sizeof(S) == 8 ? 64 : 32, 2, shape, bias ? DOCC_ROCM_BINARY_ADD : -1, shape, C, 0.0,
                                               bias ? row : nullptr, bias, 0.0, activation >= 0 ? 1 : 0, post, C);
        }
    }
    size_t lds;
    if (fin) {
        // kernels with the chain in their store: the asynchronous ones the picker chooses from, A stored by rows
        const bool built = cfg.stages > 0 && !ta && sizeof(T) <= 4 && (sizeof(T) == 4 || !cfg.spread || cfg.small) && n % 8 == 0 &&
                           ((uintptr_t) fin->bias | (uintptr_t) fin->residual | (uintptr_t) fin->out) % 16 == 0;
        if (!built) return through_memory(plain_product);
        std::snprintf(name, sizeof(name), "docc_%sa_%dx%dx%d%c%d_n%c_f", prefix, cfg.bm, cfg.bn, cfg.bk, cfg.small ? 'q' : 's', cfg.stages, tb ? 't' : 'n');
        const size_t ring = (size_t) cfg.stages * ((size_t) cfg.bm * cfg.bk + (size_t) cfg.bk * cfg.bn) * sizeof(T);
        // a wave's (of 2 x 2) rows on their way out, up to 64 of them, padded by four floats (FinishShape)
        const size_t turned = (size_t) cfg.waves * (cfg.bm / 2 < 64 ? cfg.bm / 2 : 64) * (cfg.bn / 2 + 4) * sizeof(float);
        return launch(name, (uint32_t) tiles, 1, 1, 64 * cfg.waves, (uint32_t) (ring > turned ? ring : turned), s, A, B, (long) m, (long) n, (long) k,
                      (long) lda, (long) ldb, (float) alpha, *fin);
    }
    if (cfg.stages > 0) {
        std::snprintf(name, sizeof(name), "docc_%sa_%dx%dx%d%c%d_%c%c", prefix, cfg.bm, cfg.bn, cfg.bk, cfg.small ? 'q' : cfg.spread ? 'p' : 's', cfg.stages,
                      ta ? 't' : 'n', tb ? 't' : 'n');
        lds = (size_t) cfg.stages * ((size_t) cfg.bm * cfg.bk + (size_t) cfg.bk * cfg.bn) * sizeof(T);
    } else {
        std::snprintf(name, sizeof(name), "docc_%s_%dx%dx%d_%c%c_%c", prefix, cfg.bm, cfg.bn, cfg.bk, ta ? 't' : 'n',
                      tb ? 't' : 'n', aligned ? 'a' : 'u');
        lds = gemm_lds_bytes(cfg, ta, tb, sizeof(T));
    }
    // the variants with bias / activation in the store carry the suffix "_e"
    if (bias || activation >= 0) std::strncat(name, "_e", sizeof(name) - std::strlen(name) - 1);
    if (cfg.stages > 0)
        return launch(name, (uint32_t) tiles, (uint32_t) batch, 1, 64 * cfg.waves, (uint32_t) lds, s, A, B, C, (long) m, (long) n,
                      (long) (k_total > 0 ? k_total : k), (long) lda, (long) ldb, (long) ldc, alpha, beta, bias, activation, (long) batch_a,
                      (long) batch_b, (long) batch_c, (long) (k_total > 0 ? k : 0));
    if (k_total > 0) return fail(DOCC_ROCM_ERR_UNSUPPORTED, "%s: K in parts needs the asynchronous tiles", prefix);
    return launch(name, (uint32_t) tiles, (uint32_t) batch, 1, 64 * cfg.waves, (uint32_t) lds, s, A, B, C, (long) m, (long) n,
                  (long) k, (long) lda, (long) ldb, (long) ldc, alpha, beta, bias, activation, (long) batch_a, (long) batch_b,
                  (long) batch_c);
}

} // namespace

// A batch of equally shaped products in launches of at most 65535 entries (the limit of gridDim.y).
template <typename T, typename S>
static int gemm_batched(const char* prefix, docc_rocm_stream_t stream, int trans_a, int trans_b, int64_t m, int64_t n, int64_t k,
                        S alpha, const T* A, int64_t lda, int64_t stride_a, const T* B, int64_t ldb, int64_t stride_b, S beta, S* C,
                        int64_t ldc, int64_t stride_c, int64_t batch,
                        Picker pick) {
    if (batch < 0) return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "%s: negative batch", prefix);
    const int64_t kMaxGridY = 65535;
    for (int64_t b0 = 0; b0 < batch; b0 += kMaxGridY) {
        const int64_t nb = batch - b0 < kMaxGridY ? batch - b0 : kMaxGridY;
        const int rc = gemm_launch<T, S>(prefix, stream, trans_a, trans_b, m, n, k, alpha, A ? A + b0 * stride_a : A, lda,
                                         B ? B + b0 * stride_b : B, ldb, beta, C ? C + b0 * stride_c : C, ldc, pick, nullptr, -1, nb,
                                         stride_a, stride_b, stride_c);
        if (rc) return rc;
    }
    return 0;
}

extern "C" {

// Tile selection. `force`: +1 largest tile, -1 smallest tile, 0 by problem size. `aligned`: 1 on whole vectors, 2 on lines of 128 bytes too.
// Asynchronous (staged) configurations need aligned operands; the others handle everything.
// tiles of one matrix times the number of matrices: what there is to spread over the compute units
static int64_t tiles_of(int64_t m, int64_t n, int bm, int bn, int64_t batch = 1) { return ((m + bm - 1) / bm) * ((n + bn - 1) / bn) * batch; }

static TileConfig pick_sgemm(int64_t m, int64_t n, int64_t, bool, int64_t batch, int aligned, int force, int cus) {
    const TileConfig huge{256, 256, 32, 4, 2}, wide{128, 256, 32, 4, 2}, big{128, 128, 32, 4, 3}, small{64, 64, 16, 4, 4};
    const TileConfig plain_big{128, 128, 16, 4, 0}, plain_small{64, 64, 16, 4, 0};
    if (!aligned) return force > 0 ? plain_big : force < 0 ? plain_small : (tiles_of(m, n, 128, 128, batch) >= 256 ? plain_big : plain_small);
    if (force) return force > 0 ? huge : small;
    // Score = share of a tile's area that is real output x share of the CUs that get a work-group x what the
    // tile sustains relative to the 128x256 one (146 / 141 / 138 / about 105 TFLOP/s on large problems): a 64-row
    // product wastes half of a 128-row tile, a 1000^2 one leaves most CUs idle with the large tiles.
    auto score = [&](const TileConfig& c, double rel) {
        const double padded = (double) ((m + c.bm - 1) / c.bm * c.bm) * (double) ((n + c.bn - 1) / c.bn * c.bn);
        const double fill = (double) tiles_of(m, n, c.bm, c.bn, batch) / cus;
        return rel * ((double) m * (double) n / padded) * (fill < 1.0 ? fill : 1.0);
    };
    const double sh = score(huge, 1.03), sw = score(wide, 1.0), sb = score(big, 0.97), ss = score(small, 0.75);
    // one work-group of the two largest tiles owns a CU, so their work-groups run in rounds: the 256x256 tile only
    // where its rounds take no longer than those of the 128x256 one
    auto rounds = [&](const TileConfig& c) { return (double) ((tiles_of(m, n, c.bm, c.bn, batch) + cus - 1) / cus) * c.bm * c.bn; };
    if (sh >= sw && sh >= sb && sh >= ss && rounds(huge) / 1.03 <= rounds(wide)) return huge;
    return sw >= sb && sw >= ss ? wide : sb >= ss ? big : small;
}

static TileConfig pick_dgemm(int64_t m, int64_t n, int64_t, bool, int64_t batch, int aligned, int force, int) {
    const TileConfig big{128, 128, 16, 4, 3}, mid{64, 64, 16, 4, 4}, small{64, 32, 16, 4, 4};
    const TileConfig plain_big{128, 128, 16, 4, 0}, plain_small{64, 64, 16, 4, 0};
    if (!aligned) return force > 0 ? plain_big : plain_small;
    if (force) return force > 0 ? big : small;
    const int64_t t = tiles_of(m, n, 64, 64, batch);
    return t >= 2048 ? big : t > 512 ? mid : small;   // few tiles: halve them so that two work-groups share a CU
}

static TileConfig pick_bgemm(int64_t m, int64_t n, int64_t k, bool tb, int64_t batch, int aligned, int force, int cus) {
    // big: on the 16x16x32 MFMA where K allows it (see gemm_launch), else on the 32x32x16 one with the copies dealt out
    const TileConfig big{256, 256, 32, 4, 4, true, true}, wide{128, 256, 64, 4, 3}, deep{128, 128, 64, 4, 4}, small{128, 128, 32, 4, 4};
    const TileConfig plain_big{256, 256, 64, 4, 0}, plain_small{128, 128, 64, 4, 0};
    if (!aligned) return force > 0 ? plain_big : force < 0 ? plain_small : (tiles_of(m, n, 256, 256, batch) >= 256 ? plain_big : plain_small);
    if (force) return force > 0 ? big : small;
    const TileConfig* best = &big;
    double least = bgemm_seconds(big, m, n, k, tb, batch, cus, aligned == 2);
    for (const TileConfig* c : {&wide, &deep, &small}) {
        const double t = bgemm_seconds(*c, m, n, k, tb, batch, cus, aligned == 2);
        if (t < least) {
            least = t;
            best = c;
        }
    }
    return *best;
}

int docc_rocm_sgemm(docc_rocm_stream_t stream, int trans_a, int trans_b, int64_t m, int64_t n, int64_t k, float alpha,
                    const float* A, int64_t lda, const float* B, int64_t ldb, float beta, float* C, int64_t ldc) {
    return gemm_launch<float>("sgemm", stream, trans_a, trans_b, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, pick_sgemm);
}

int docc_rocm_dgemm(docc_rocm_stream_t stream, int trans_a, int trans_b, int64_t m, int64_t n, int64_t k,
                    double alpha, const double* A, int64_t lda, const double* B, int64_t ldb, double beta, double* C,
                    int64_t ldc) {
    return gemm_launch<double>("dgemm", stream, trans_a, trans_b, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, pick_dgemm);
}

int docc_rocm_bf16gemm_f32(docc_rocm_stream_t stream, int trans_a, int trans_b, int64_t m, int64_t n, int64_t k,
                           float alpha, const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb, float beta,
                           float* C, int64_t ldc) {
    return gemm_launch<uint16_t, float>("bgemm", stream, trans_a, trans_b, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc,
                                        pick_bgemm);
}

int docc_rocm_sgemm_epilogue(docc_rocm_stream_t stream, int trans_a, int trans_b, int64_t m, int64_t n, int64_t k, float alpha,
                             const float* A, int64_t lda, const float* B, int64_t ldb, float beta, float* C, int64_t ldc,
                             const float* bias, int activation) {
    return gemm_launch<float>("sgemm", stream, trans_a, trans_b, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, pick_sgemm, bias,
                              activation);
}

int docc_rocm_dgemm_epilogue(docc_rocm_stream_t stream, int trans_a, int trans_b, int64_t m, int64_t n, int64_t k,
                             double alpha, const double* A, int64_t lda, const double* B, int64_t ldb, double beta, double* C,
                             int64_t ldc, const double* bias, int activation) {
    return gemm_launch<double>("dgemm", stream, trans_a, trans_b, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, pick_dgemm, bias,
                               activation);
}

int docc_rocm_bf16gemm_f32_epilogue(docc_rocm_stream_t stream, int trans_a, int trans_b, int64_t m, int64_t n, int64_t k,
                                    float alpha, const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb, float beta,
                                    float* C, int64_t ldc, const float* bias, int activation) {
    return gemm_launch<uint16_t, float>("bgemm", stream, trans_a, trans_b, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc,
                                        pick_bgemm, bias, activation);
}

// the chain behind a product as the kernels take it, from the launchers' arguments
static int linear_finish(int type, int64_t m, int64_t n, const void* bias, int bias_type, int activation, const void* residual, int residual_type, int rounding, void* Y,
                         int y_type, LinearFinish* finish) {
    auto is = [](int t, int a, int b) { return t == a || t == b; };
    if (!is(type, DOCC_ROCM_TYPE_F32, DOCC_ROCM_TYPE_BF16) || !is(y_type, DOCC_ROCM_TYPE_F32, DOCC_ROCM_TYPE_BF16) ||
        (bias && !is(bias_type, DOCC_ROCM_TYPE_F32, DOCC_ROCM_TYPE_BF16)) || (residual && !is(residual_type, DOCC_ROCM_TYPE_F32, DOCC_ROCM_TYPE_BF16)))
        return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "linear: operands are float32 or bf16");
    if (activation != -1 && activation != DOCC_ROCM_UNARY_ABS && activation != DOCC_ROCM_UNARY_RELU && activation != DOCC_ROCM_UNARY_SIGMOID &&
        activation != DOCC_ROCM_UNARY_TANH && !(activation >= DOCC_ROCM_ACT_GELU && activation <= DOCC_ROCM_ACT_SILU))
        return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "linear: unknown activation %d", activation);
    if (rounding & ~(DOCC_ROCM_ROUND_BEFORE_ACT | DOCC_ROCM_ROUND_AFTER_ACT)) return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "linear: unknown rounding %d", rounding);
    if (m > 0 && n > 0 && !Y) return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "linear: null pointer");
    LinearFinish& f = *finish;
    f = LinearFinish{bias, residual, Y, 0, activation};
    if (bias && bias_type == DOCC_ROCM_TYPE_BF16) f.flags |= kBiasBf16;
    if (residual && residual_type == DOCC_ROCM_TYPE_BF16) f.flags |= kResidualBf16;
    if (y_type == DOCC_ROCM_TYPE_BF16) f.flags |= kOutBf16;
    if (rounding & DOCC_ROCM_ROUND_BEFORE_ACT) f.flags |= kRoundBeforeAct;
    if (rounding & DOCC_ROCM_ROUND_AFTER_ACT) f.flags |= kRoundAfterAct;
    return 0;
}

int docc_rocm_linear(docc_rocm_stream_t stream, int type, int trans_a, int trans_b, int64_t m, int64_t n, int64_t k, float alpha, const void* A,
                     int64_t lda, const void* B, int64_t ldb, const void* bias, int bias_type, int activation, const void* residual,
                     int residual_type, int rounding, void* Y, int y_type) {
    LinearFinish f{};
    if (int rc = linear_finish(type, m, n, bias, bias_type, activation, residual, residual_type, rounding, Y, y_type, &f)) return rc;
    if (type == DOCC_ROCM_TYPE_F32)
        return gemm_launch<float>("sgemm", stream, trans_a, trans_b, m, n, k, alpha, (const float*) A, lda, (const float*) B, ldb, 0.0f, (float*) nullptr, n,
                                  pick_sgemm, (const float*) nullptr, -1, 1, 0, 0, 0, &f);
    return gemm_launch<uint16_t, float>("bgemm", stream, trans_a, trans_b, m, n, k, alpha, (const uint16_t*) A, lda, (const uint16_t*) B, ldb, 0.0f,
                                        (float*) nullptr, n, pick_bgemm, (const float*) nullptr, -1, 1, 0, 0, 0, &f);
}

int docc_rocm_norm_linear(docc_rocm_stream_t stream, int type, int64_t m, int64_t n, int64_t k, float eps, const void* X, const void* weight, const void* norm_bias,
                          float alpha, const void* B, int64_t ldb, const void* bias, int bias_type, int activation, const void* residual, int residual_type, int rounding,
                          void* scratch, void* Y, int y_type) {
    LinearFinish f{};
    if (int rc = linear_finish(type, m, n, bias, bias_type, activation, residual, residual_type, rounding, Y, y_type, &f)) return rc;
    if (m < 0 || n < 0 || k < 0 || ldb < (k > 1 ? k : 1)) return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "norm_linear: bad shape");
    if (m == 0 || n == 0) return 0;
    // Rows that a wavefront holds, every work-group's in LDS (csrc/kernels/gemm_waves.hip): a launch of 3 to 4 us less. Every work-group normalises all rows again,
    // 4 to 16 vectors a lane, while it waits for its first pieces of B. DOCC_ROCM_GEMM_WAVES=0 or a tile other than 16 keeps the layer norm a launch of its own
    // (tests, tuning).
    const char* env = gemm_tuning_set() ? std::getenv("DOCC_ROCM_GEMM_WAVES") : nullptr;
    const int forced = env ? std::atoi(env) : -1;
    const bool bf16 = type == DOCC_ROCM_TYPE_BF16;
    const int64_t v = bf16 ? 8 : 4;
    const int rows = m <= 8 ? 8 : 16, vectors = k <= 256 * v ? 4 : 8;      // vectors a lane holds
    // Two launches read X and the norm's operands before the first store to Y, and what lies in `scratch` behind the norm's store: one launch reads X while it
    // stores Y, and stores no `scratch`.
    auto meet = [](const void* p, int64_t p_bytes, const void* q, int64_t q_bytes) {
        return p && q && (uintptr_t) p < (uintptr_t) q + (uintptr_t) q_bytes && (uintptr_t) q < (uintptr_t) p + (uintptr_t) p_bytes;
    };
    const int64_t e = bf16 ? 2 : 4, x_bytes = m * k * e, y_bytes = m * n * (f.flags & kOutBf16 ? 2 : 4);
    const bool apart = !meet(X, x_bytes, Y, y_bytes) && !meet(weight, k * e, Y, y_bytes) && !meet(norm_bias, k * e, Y, y_bytes) &&
                       !meet(scratch, x_bytes, residual, m * n * (f.flags & kResidualBf16 ? 2 : 4)) && !meet(scratch, x_bytes, B, ((n - 1) * ldb + k) * e) &&
                       !meet(scratch, x_bytes, bias, n * (f.flags & kBiasBf16 ? 2 : 4));
    if (apart && m <= 16 && k >= 8 * v && k <= 512 * v && (rows == 8 || vectors == 4) && n % 8 == 0 && waves_shape_ok(m, n, k, k, ldb, true, bf16 ? 2 : 4) && alpha != 0.0f && X && B &&
        (forced < 0 || forced == 16) &&
        ((uintptr_t) X | (uintptr_t) weight | (uintptr_t) norm_bias | (uintptr_t) B | (uintptr_t) bias | (uintptr_t) residual | (uintptr_t) Y) % 16 == 0) {
        if (int rc = ensure_device()) return rc;
        // the rings, the rows, and a piece's length behind the last
        const int64_t groups = (n + 15) / 16, lds = 8 * 2 * 16 * 128 + rows * (k + v) * (bf16 ? 2 : 4) + 128;
        // all work-groups at once: the next ones would normalise the rows again with nothing to hide that behind
        const int64_t at_once = (!bf16 || (vectors == 4 && rows == 8)) && 2 * lds <= 160 * 1024 ? 2 : 1;
        if (lds <= 160 * 1024 && (forced > 0 || groups <= at_once * cu_count())) {
            const struct {
                const void *weight, *bias;
                float eps;
            } norm{weight, norm_bias, eps};
            char name[64];
            std::snprintf(name, sizeof(name), "docc_%cgemm_waves_norm%d_m%d_f", bf16 ? 'b' : 's', vectors, rows);
            return launch(name, (uint32_t) groups, 1, 1, 512, (uint32_t) lds, (hipStream_t) stream, X, (long) k, B, (long) ldb, (long) m, (long) n, (long) k, alpha, f, norm);
        }
    }
    if (!scratch && k > 0) return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "norm_linear: null pointer");
    if (int rc = docc_rocm_layer_norm(stream, type, m, k, eps, X, weight, norm_bias, scratch)) return rc;
    return docc_rocm_linear(stream, type, DOCC_ROCM_NO_TRANS, DOCC_ROCM_TRANS, m, n, k, alpha, scratch, k > 1 ? k : 1, B, ldb, bias, bias_type, activation, residual,
                            residual_type, rounding, Y, y_type);
}

int docc_rocm_sgemm_batched(docc_rocm_stream_t stream, int trans_a, int trans_b, int64_t m, int64_t n, int64_t k, float alpha,
                            const float* A, int64_t lda, int64_t stride_a, const float* B, int64_t ldb, int64_t stride_b, float beta,
                            float* C, int64_t ldc, int64_t stride_c, int64_t batch) {
    return gemm_batched<float, float>("sgemm", stream, trans_a, trans_b, m, n, k, alpha, A, lda, stride_a, B, ldb, stride_b, beta, C,
                                      ldc, stride_c, batch, pick_sgemm);
}

int docc_rocm_dgemm_batched(docc_rocm_stream_t stream, int trans_a, int trans_b, int64_t m, int64_t n, int64_t k, double alpha,
                            const double* A, int64_t lda, int64_t stride_a, const double* B, int64_t ldb, int64_t stride_b,
                            double beta, double* C, int64_t ldc, int64_t stride_c, int64_t batch) {
    return gemm_batched<double, double>("dgemm", stream, trans_a, trans_b, m, n, k, alpha, A, lda, stride_a, B, ldb, stride_b, beta,
                                        C, ldc, stride_c, batch, pick_dgemm);
}

int docc_rocm_bf16gemm_f32_batched(docc_rocm_stream_t stream, int trans_a, int trans_b, int64_t m, int64_t n, int64_t k, float alpha,
                                   const uint16_t* A, int64_t lda, int64_t stride_a, const uint16_t* B, int64_t ldb,
                                   int64_t stride_b, float beta, float* C, int64_t ldc, int64_t stride_c, int64_t batch) {
    return gemm_batched<uint16_t, float>("bgemm", stream, trans_a, trans_b, m, n, k, alpha, A, lda, stride_a, B, ldb, stride_b, beta,
                                         C, ldc, stride_c, batch, pick_bgemm);
}

} // extern "C"
