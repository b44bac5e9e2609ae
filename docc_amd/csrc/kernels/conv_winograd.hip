// ml::Conv, 2-d NCHW fp32, 3x3 without dilation and with steps of one or two, by Winograd's minimal filtering F(2x2, 3x3)
// (S. Winograd, Arithmetic Complexity of Computations, 1980; A. Lavin and S. Gray, Fast Algorithms for Convolutional
// Neural Networks, 2016): a 2x2 tile of outputs is A^T [ sum over channels of (G g G^T) .* (B^T d B) ] A of the 4x4 input pixels d
// around it, 16 products a channel instead of 36.
//
// Steps of two: a 2x2 tile of outputs reads 5x5 pixels. Along an axis taps 0 and 2 meet the pixels 0, 2 and 4, a two-tap filter with two outputs: (x0 - x2) w0,
// x2 (w0 + w2), (x4 - x2) w2; tap 1 meets x1 and x3. Five products for six, 25 for 36 in two axes, and as the products that go to one output alone
// share a sum with those of tap 1, nine sums (and four, see below). The filters have 16 components again, so that their way is the same.
//
// What bounds the direct form is the fp32 matrix pipe (one work-group of docc_conv2d_f32_halo_* keeps it at two thirds of its peak); the 16
// sums over the channels are the same matrix product of 16 / 36 of the size, and everything else a tile needs fits beside
// it: fp32 MFMAs are long (32 cycles the 16x16x4 form), 32 additions and 16 loads a lane are issued under 32 of them.
//
// Work-group: 64 * NW threads, 32 output channels x 16 * NW tiles. A wave takes 16 tiles and all 16 components: lane l holds
// tile l % 16 and channel l / 16 of a step of four channels, which is the B operand of v_mfma_f32_16x16x4_f32, so the
// transformed input never leaves the registers that it is computed in, and neither do the sums: component by component they
// lie in the same lane and register, and the output transform is additions of registers. The filters go through LDS: per chunk of eight channels
// every thread transforms 4 / NW of the 32 x 8 filters and writes their 16 components, quads of components apart, so that a lane reads the A
// operands of four components with 128 bits; two buffers, one barrier per chunk.
//
// The input comes by buffer loads: a row above or below the image (or of a tile beyond the last one) has an offset beyond the buffer's end,
// for which the load gives 0, and the channel is the scalar offset.
//
// What bounds it now is the issue of everything that is no MFMA: such an instruction takes some five cycles of the wave and is only partly hidden
// by the other wave of the SIMD. Measured on 166 x 256 x 14 x 14 -> 256 (four work-groups a CU): 150 us = 257 TFLOP/s of the direct form's count; the MFMAs
// alone 124 us, without the filters' way 141, without loading pixels 135. Interleaved one MFMA, two others it took 179 us, the others in one run amid
// eight MFMAs 164, and with fewer of them (vector loads of a row instead of its pixels, no factors of one half, buffers by constant
// offsets) the 150. Against the direct form: 32 x 64 x 56 x 56 -> 64 71 -> 48 us, 32 x 256 x 14 x 14 -> 256 92 -> 48; steps of
// two: 50 x 80 x 52 x 52 -> 160 153 -> 57, 3 x 448 x 51 x 51 -> 896 257 -> 106 (its MFMAs 1.52 us a chunk and work-group, measured 1.6). Pixel by pixel a row's loads touch
// their cache lines once each, which bounds steps of two: 12 x 96 x 8 x 8 51 us for 25 with vectors or pairs.
//
// Rounding: the chain of additions has C terms instead of 9 C (steps of two: 3 C at most, with four sums more), the transforms add their own. An output's error is
// bounded by the sum over the channels of the largest filter value times the largest pixel of its window, that of a direct sum by the products of its own taps: where
// a few values are far larger than the others, or most are zero, the direct sum is the closer one. Relative error (2-norm) against 64 bits in units of the direct
// form's with its channels in as many parts, 4 x C x 28 x 28, steps of one / two:
//                                             C = 8        16          32          64 (both in parts)   512 (both in parts)
//   N(0, 1)                                   0.91 / 0.95  0.77 / 0.87 0.68 / 0.82    0.78 / 0.89       0.70 / 0.89
//   its positive part                         1.10 / 1.00  0.96 / 0.92 0.85 / 0.85    0.92 / 0.90       0.86 / 0.95
//   that with half of the rest zero           1.48 / 1.24  1.25 / 1.12 1.10 / 1.02    1.20 / 1.08       1.07 / 1.07
// Filters with one value that is not zero have exact direct sums; here 5e-8 of the result is lost with steps of one. Images with one value of a hundred 1e4 times as
// large: 0.7 to 0.9 of the direct form's error as a whole, but the worst output, as a share of the sum of its taps' magnitudes, 40 times it at C = 32, 16 at 64, 1.5 at
// 256. So the launcher takes this form from 32 channels on, and with no longer chains than keep the positive part's error at the direct form's (winograd_longest() in
// csrc/rt/ops_conv.cpp): 90 drawn layers (1-64 images, 32-512 channels, 7 x 7 to 64 x 64) 0.68 / 0.80 of it on N(0, 1), 0.83 / 0.82 on the positive part
// (geometric means; 1.05 and 1.02 at most). An output depends on the pixels of its own window alone, as in the direct form, but where
// products cancel (or a sum of pixels overflows) an infinity can come out as a NaN: a wavefront with outputs that are not finite sums its own again, directly.
#include "elementwise_ops.h"
#include "conv_params.h"
#include <type_traits>

namespace docc_k {

typedef float wf4 __attribute__((ext_vector_type(4)));
typedef float wf2 __attribute__((ext_vector_type(2)));

// How a lane loads the pixels of a row:
//   kPixels   one by one, each with an offset of its own; any padding
//   kVector   four as one vector, with steps of two the column before them apart. One column of padding: only the outer columns can lie in it. The
//             vector reads a neighbouring row's pixels there, which are dropped after the row transform; work-groups with a tile for which they lie
//             outside the tensor load pixel by pixel. With steps of two rows are whole vectors and nothing of the kind happens.
//   kVectorOdd  (steps of one) the same for rows of odd length, whose last tile has two columns in the padding
//   kPairs    (steps of two) the column before, then two pairs. Of a pair that begins with the row's last pixel the one before is loaded and shifted.
enum WinogradLoads { kPixels, kVector, kVectorOdd, kPairs };

template <int S>
struct ConvWinograd {
    static constexpr int NW = 4;                   // waves
    static constexpr int CI = 8;                   // channels per chunk
    static constexpr int CS = 4 * 128 + 4;         // floats from one channel's components in LDS to the next's (eight lanes write a channel each: a vector further)
    static constexpr int STAGE = CI * CS;
    static constexpr int RAW = 32 * CI * 9;        // filters of a chunk as they lie in memory
    static constexpr int PX = S == 1 ? 4 : 5;      // pixels a tile reads along a row or column
    static constexpr int RG = PX;                  // rows of products per channel
    static constexpr int NA = S == 1 ? 4 : 3;      // rows of sums
    // the row of filter components and the row of sums that row i of products goes with
    static constexpr int filter_row(int i) { return i == 4 ? 3 : i; }
    static constexpr int sum_row(int i) { return S == 1 ? i : i == 3 ? 0 : i == 4 ? 2 : i; }
    // Where four products would share a sum, the one that is a difference of pixels in both axes, the largest, has a sum of its own that is added at the end: with nine
    // sums the error on N(0, 1) images was the direct form's (64 to 512 channels 1.00), with thirteen it is 0.89 of it, in the same time.
    static constexpr int NS = S == 1 ? 16 : 13;
    static constexpr int sum_of(int i, int j) {
        const bool corner = S == 2 && (i == 0 || i == 2) && (j == 0 || j == 2);
        return corner ? NA * NA + i + j / 2 : NA * sum_row(i) + sum_row(j);
    }
    static constexpr int WL = (RAW / 4 + 64 * NW - 1) / (64 * NW);   // vectors of them a thread moves
    static constexpr int LDS_FLOATS = 2 * STAGE + 2 * RAW + 4;

    // where a lane's tile lies, and the work-group's operands as buffers: X from its first image n0 on and the filters from oc0 on; the launcher has seen to it that
    // what a work-group addresses takes less than 2^30 bytes. (X four pixels early: the column before an image's first one has an offset as well.)
    static constexpr int kEarly = 4;
    static constexpr int kNone = (int) 0x80000000;      // an offset beyond either: the load gives 0
    typedef decltype(__builtin_amdgcn_make_buffer_rsrc((void*) nullptr, 0, 0, 0)) buffer_t;
    struct Place {
        bool ok;
        int n0, n, oh, ow, ih0, iw0;
        buffer_t xbuf, wbuf;
        __device__ __forceinline__ Place(const ConvParams& p, int tid, int tile0, int oc0, int c0) {
            const int TW = (p.OW + 1) >> 1, per_image = ((p.OH + 1) >> 1) * TW;
            const int tile = tile0 + (tid >> 6) * 16 + (tid & 15);
            ok = tile < p.N * per_image;
            n0 = tile0 / per_image;
            const int rest = (ok ? tile : tile0) % per_image;
            n = (ok ? tile : tile0) / per_image;
            oh = 2 * (rest / TW), ow = 2 * (rest % TW);
            ih0 = S * oh - p.pad_h, iw0 = S * ow - p.pad_w;
            const long left = ((long) (p.N - n0) * p.XC * p.H * p.W - (long) c0 * p.H * p.W + kEarly) * 4;
            xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.X) + (((long) n0 * p.XC + c0) * p.H * p.W - kEarly), 0,
                                                     (int) (left < 0x7fffffffL ? left : 0x7fffffffL), 0x00020000);
            const long wleft = ((long) (p.OC - oc0) * p.C - c0) * 36;
            wbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.Wt) + ((long) oc0 * p.C + c0) * 9, 0,
                                                     (int) (wleft < 0x7fffffffL ? wleft : 0x7fffffffL), 0x00020000);
        }
    };

    // channels [c0, c0 + 8 * chunks) of X and Wt; the work-group's tiles from tile0 on, output channels from oc0 on
    template <int LOADS>
    static __device__ __forceinline__ void run(const ConvParams& p, const ConvFinish& fin, float* lds, int tile0, int oc0, int c0, int chunks) {
        const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
        const int l16 = lane & 15, lk = lane >> 4;
        const Place place(p, tid, tile0, oc0, c0);
        const bool tile_ok = place.ok;
        const int n0 = place.n0, n = place.n, ow = place.ow, ih0 = place.ih0, iw0 = place.iw0;
        const buffer_t xbuf = place.xbuf, wbuf = place.wbuf;
        const int HW4 = p.H * p.W * 4;

        const bool first_col = ow == 0, odd_col = ow + 1 >= p.W, last_col = ow + 2 >= p.W;   // kVector, kVectorOdd: columns 0, 2 and 3 in the padding
        constexpr int NOFF = LOADS == kPixels ? PX : LOADS == kPairs ? 3 : S;
        int voff[PX][NOFF];
        bool shifted[2] = {false, false};
#pragma unroll
        for (int r = 0; r < PX; r++)
#pragma unroll
            for (int c = 0; c < NOFF; c++) {
                const int ih = ih0 + r;
                int iw = iw0 + (LOADS == kPairs && c > 0 ? 2 * c - 1 : c);
                bool in = tile_ok && ih >= 0 && ih < p.H && ((LOADS != kPixels && LOADS != kPairs && S == 1) || (iw >= 0 && iw < p.W));
                if (LOADS == kPairs && c > 0) {
                    // (the launcher takes no padding for which a pair begins with the column before the first)
                    if (iw == p.W - 1) shifted[c - 1] = true, iw--;
                    in = tile_ok && ih >= 0 && ih < p.H && iw >= 0 && iw + 1 < p.W;
                }
                voff[r][c] = in ? ((n - n0) * p.XC * p.H * p.W + (lk * p.H + ih) * p.W + iw + kEarly) * 4 : kNone;
            }
        float d[2][PX][PX];
        auto xload = [&](int step, int r, int to) {
            const int at = step * 4 * HW4;
            auto one = [&](int c, int off) { d[to][r][c] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xbuf, voff[r][off], at, 0)); };
            if constexpr (LOADS == kVector || LOADS == kVectorOdd) {
                const wf4 x = __builtin_bit_cast(wf4, __builtin_amdgcn_raw_buffer_load_b128(xbuf, voff[r][S - 1], at, 0));
#pragma unroll
                for (int c = 0; c < 4; c++) d[to][r][S - 1 + c] = x[c];
                if constexpr (S == 2) one(0, 0);
            } else if constexpr (LOADS == kPairs) {
                one(0, 0);
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const wf2 x = __builtin_bit_cast(wf2, __builtin_amdgcn_raw_buffer_load_b64(xbuf, voff[r][1 + q], at, 0));
                    d[to][r][1 + 2 * q] = x[0], d[to][r][2 + 2 * q] = x[1];
                }
            } else {
#pragma unroll
                for (int c = 0; c < PX; c++) one(c, c);
            }
        };

        // The filters' way: vectors of a chunk as they lie in memory ([output channel][channel][tap], 288 bytes of a row) to registers and to
        // LDS, from there nine values to the thread that transforms them, 16 components back to LDS.
        float* const raw = lds + 2 * STAGE;
        int woff[WL];
        float* wdst[WL];
#pragma unroll
        for (int u = 0; u < WL; u++) {
            const int v = tid + u * 64 * NW, row = v / (CI * 9 / 4);
            const bool in = v < RAW / 4;
            woff[u] = in && oc0 + row < p.OC ? (row * p.C * 9 + (v % (CI * 9 / 4)) * 4) * 4 : kNone;
            wdst[u] = in ? raw + v * 4 : raw + 2 * RAW;        // (surplus threads of the last round: a spare vector)
        }
        wf4 wr[WL];
        auto wload = [&](int chunk) {
#pragma unroll
            for (int u = 0; u < WL; u++) wr[u] = __builtin_bit_cast(wf4, __builtin_amdgcn_raw_buffer_load_b128(wbuf, woff[u], chunk * (CI * 36), 0));
        };
        auto wraw = [&](int buf, int u) {
            const bool spare = (u + 1) * 64 * NW > RAW / 4;    // the round with surplus threads: their vector is not moved between the buffers
            *reinterpret_cast<wf4*>(wdst[u] + (spare && buf && tid + u * 64 * NW >= RAW / 4 ? 0 : buf * RAW)) = wr[u];
        };
        const int uc = tid & 7, uo = tid >> 3;
        float g[9];
        const float* const gsrc = raw + uo * (CI * 9) + uc * 9;
        auto gread = [&](int buf) {
#pragma unroll
            for (int t = 0; t < 9; t++) g[t] = gsrc[buf * RAW + t];
        };
        float* const udst = lds + uc * CS + uo * 4;
        auto ustage = [&](int buf, int i) {      // row i of the components
            float h[3];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const float a = g[c], b = g[3 + c], e = g[6 + c];
                if constexpr (S == 1) h[c] = i == 0 ? a : i == 3 ? e : i == 1 ? (a + e) + b : (a + e) - b;   // (without G's halves: the output transform has them)
                else h[c] = i == 0 ? a : i == 1 ? a + e : i == 2 ? e : b;
            }
            const float s = h[0] + h[2];
            wf4 u;
            if constexpr (S == 1) u = wf4{h[0], s + h[1], s - h[1], h[2]};
            else u = wf4{h[0], s, h[2], h[1]};
            *reinterpret_cast<wf4*>(udst + buf * STAGE + i * 128) = u;
        };

        wf4 acc[NS][2];
        const float* const ulane = lds + lk * CS + l16 * 4;
        wf4 a[2][2];
        auto aread = [&](int buf, int half, int f) {      // row f of the filter components
#pragma unroll
            for (int o = 0; o < 2; o++) a[f & 1][o] = *reinterpret_cast<const wf4*>(ulane + buf * STAGE + half * (4 * CS) + f * 128 + o * 64);
        };
        // the transformed pixels of row i of the products
        float v[2][RG];
        auto vrow = [&](float (&x)[PX][PX], int i, int to) {
            float t[PX];
#pragma unroll
            for (int c = 0; c < PX; c++) {
                if constexpr (S == 1) t[c] = i == 0 ? x[0][c] - x[2][c] : i == 1 ? x[1][c] + x[2][c] : i == 2 ? x[2][c] - x[1][c] : x[1][c] - x[3][c];
                else t[c] = i == 0 ? x[0][c] - x[2][c] : i == 1 ? x[2][c] : i == 2 ? x[4][c] - x[2][c] : i == 3 ? x[1][c] : x[3][c];
            }
            if constexpr (S == 1) {
                if constexpr (LOADS != kPixels) {
                    t[0] = first_col ? 0.f : t[0];
                    if constexpr (LOADS == kVectorOdd) t[2] = odd_col ? 0.f : t[2];
                    t[3] = last_col ? 0.f : t[3];
                }
                v[to][0] = t[0] - t[2], v[to][1] = t[1] + t[2], v[to][2] = t[2] - t[1], v[to][3] = t[1] - t[3];
            } else {
                if constexpr (LOADS == kPairs) {
#pragma unroll
                    for (int q = 0; q < 2; q++) {
                        t[1 + 2 * q] = shifted[q] ? t[2 + 2 * q] : t[1 + 2 * q];
                        t[2 + 2 * q] = shifted[q] ? 0.f : t[2 + 2 * q];
                    }
                }
                v[to][0] = t[0] - t[2], v[to][1] = t[2], v[to][2] = t[4] - t[2], v[to][3] = t[1], v[to][4] = t[3];
            }
        };
        auto mfmas = [&](int i, int from) {
            const int f = filter_row(i);
#pragma unroll
            for (int j = 0; j < RG; j++)
#pragma unroll
                for (int o = 0; o < 2; o++) {
                    wf4& sum = acc[sum_of(i, j)][o];
                    sum = __builtin_amdgcn_mfma_f32_16x16x4f32(a[f & 1][o][filter_row(j)], v[from][j], sum, 0, 0, 0);
                }
        };
        // Each row of products is a scheduling region: its MFMAs, between them the operands of the next row (filters from LDS,
        // pixels transformed), the loads that refill the pixel registers that are free, and filters.
        auto shape = [&]() {
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);     // LDS reads
            __builtin_amdgcn_sched_group_barrier(0x008, RG, 0);    // MFMA
            __builtin_amdgcn_sched_group_barrier(0x020, 16, 0);    // loads
            __builtin_amdgcn_sched_group_barrier(0x002, 40, 0);    // VALU
            __builtin_amdgcn_sched_group_barrier(0x200, 4, 0);     // LDS writes
            __builtin_amdgcn_sched_group_barrier(0x008, RG, 0);
            __builtin_amdgcn_sched_barrier(0);
        };

        // chunk 0's filters all the way, chunk 1's as far as the registers, chunk 2's on their way
        const int last = chunks - 1;
        wload(0);
#pragma unroll
        for (int r = 0; r < PX; r++) xload(0, r, 0);
#pragma unroll
        for (int r = 0; r < PX; r++)
            if (r != 3 || S == 1) xload(1, r, 1);
#pragma unroll
        for (int u = 0; u < WL; u++) wraw(0, u);
        wload(last < 1 ? last : 1);
        __syncthreads();
        gread(0);
#pragma unroll
        for (int u = 0; u < WL; u++) wraw(1, u);
        wload(last < 2 ? last : 2);
#pragma unroll
        for (int i = 0; i < 4; i++) ustage(0, i);
        vrow(d[0], 0, 0);
        __syncthreads();
        gread(1);
        aread(0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < NS; q++)
#pragma unroll
            for (int o = 0; o < 2; o++) acc[q][o] = wf4{0.f, 0.f, 0.f, 0.f};
        // In chunk ch the filters of ch + 1 are transformed into the other buffer, those of ch + 2 written to LDS as they are, those of ch + 3
        // loaded. The barrier stands before the last row of a chunk, whose operands are in registers by then: the first ones of the next
        // chunk are read under it. (The last chunks load and stage once more what nobody reads.)
        auto chunk = [&](int ch, auto buf_c) {
            constexpr int buf = decltype(buf_c)::value;
            const int s2 = ch < last ? 2 * ch + 2 : 2 * ch, s3 = s2 + 1, w3 = ch + 3 < last ? ch + 3 : last;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int i = 0; i < RG; i++) {
                    const bool ends = i + 1 == RG;
                    if (h == 1 && ends) {
                        __syncthreads();
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    const int ni = ends ? 0 : i + 1, nh = ends ? h ^ 1 : h;
                    if (ends || filter_row(ni) != filter_row(i)) aread(ends && h == 1 ? buf ^ 1 : buf, nh, filter_row(ni));
                    vrow(d[nh], ni, (h * RG + i + 1) & 1);
                    if (h == 0 && i < 4) ustage(buf ^ 1, i);
                    if (h == 1 && i == 1) {
#pragma unroll
                        for (int u = 0; u < WL; u++) wraw(buf, u);
                        wload(w3);
                    }
                    if (h == 1 && ends) gread(buf);
                    // the pixels of two steps on, each row once this step has transformed it for the last time
                    if constexpr (S == 1) {
                        const int s = h ? s3 : s2;
                        if (i == 0) xload(s, 0, h);
                        if (i == 2) xload(s, 2, h);
                        if (i == 3) xload(s, 1, h);
                        if (i == 3 && h == 1) xload(s, 3, h);
                        if (i == 0 && h == 1) xload(s2, 3, 0);
                    } else {
                        const int s = h ? s3 : s2;
                        if (i == 0) xload(s, 0, h);
                        if (i == 2) xload(s, 2, h);
                        if (i == 3) xload(s, 4, h);
                        if (i == 4) xload(s, 1, h);
                        if (i == 0) xload(h ? s2 : 2 * ch + 1, 3, h ^ 1);
                    }
                    mfmas(i, (h * RG + i) & 1);
                    shape();
                }
        };
        int ch = 0;
        for (; ch + 1 < chunks; ch += 2) {
            chunk(ch, std::integral_constant<int, 0>{});
            chunk(ch + 1, std::integral_constant<int, 1>{});
        }
        if (ch < chunks) chunk(ch, std::integral_constant<int, 0>{});

        // (worked out again, where the tile lies: what is kept for this would take registers from the chunks)
        int tid_again = tid;
        asm volatile("" : "+v"(tid_again));
        finish(p, fin, acc, tid_again, tile0, oc0, c0, chunks);
    }

    static __device__ __forceinline__ void finish(const ConvParams& p, const ConvFinish& fin, wf4 (&acc)[NS][2], int tid, int tile0, int oc0, int c0, int chunks) {
        const int l16 = tid & 15, lk = (tid >> 4) & 3;
        const Place place(p, tid, tile0, oc0, c0);
        const bool tile_ok = place.ok;
        const int n = place.n, oh = place.oh, ow = place.ow;
        if constexpr (S == 2) {
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int o = 0; o < 2; o++) acc[q / 2 * 2 * NA + q % 2 * 2][o] += acc[NA * NA + q][o];
        }
        // outputs: rows of A^T = (1 1 1 0), (0 1 -1 -1) on both sides, the middle components halved; strides of two (1 1 0), (0 1 1)
        const long plane = (long) p.OH * p.OW;
        const bool right = ow + 1 < p.OW, below = oh + 1 < p.OH;
        const bool pairs = (p.OW & 1) == 0 && (((uintptr_t) p.Y | (uintptr_t) fin.residual) & 7) == 0;
        const long at = ((long) n * p.YC) * plane + (long) oh * p.OW + ow;
        float* const ytile = p.Y + at;
        const float* const rtile = fin.residual + at;
        float bias[2][4];
#pragma unroll
        for (int o = 0; o < 2; o++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int oc = oc0 + o * 16 + 4 * lk + r;
                bias[o][r] = p.bias ? p.bias[oc < p.OC ? oc : p.OC - 1] : -0.f;
            }
        unsigned again = 0;      // outputs that are not finite: bit 16 * o + 4 * r + 2 * row + column
        typedef float f2 __attribute__((ext_vector_type(2)));
        auto outputs = [&](auto fast_c, auto residual_c) {
            constexpr bool FAST = decltype(fast_c)::value, RESIDUAL = decltype(residual_c)::value;
            f2 res[2][4][2];         // all of them on their way before the first is needed
#pragma unroll
            for (int o = 0; o < 2; o++)
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        res[o][r][i] = f2{-0.f, -0.f};
                        if constexpr (RESIDUAL) {
                            const int oc = oc0 + o * 16 + 4 * lk + r;
                            const float* from = rtile + oc * plane + i * p.OW;
                            if constexpr (FAST) {
                                res[o][r][i] = *reinterpret_cast<const f2*>(from);
                            } else if (oc < p.OC && (i == 0 || below)) {
                                res[o][r][i][0] = from[0];
                                if (right) res[o][r][i][1] = from[1];
                            }
                        }
                    }
#pragma unroll
            for (int o = 0; o < 2; o++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int oc = oc0 + o * 16 + 4 * lk + r;
                    float s[2][NA];
#pragma unroll
                    for (int j = 0; j < NA; j++) {
                        const float m0 = acc[j][o][r], m1 = acc[NA + j][o][r], m2 = acc[2 * NA + j][o][r];
                        if constexpr (S == 1) {
                            s[0][j] = __builtin_fmaf(0.5f, m1 + m2, m0);
                            s[1][j] = __builtin_fmaf(0.5f, m1 - m2, -acc[12 + j][o][r]);
                        } else {
                            s[0][j] = m0 + m1;
                            s[1][j] = m1 + m2;
                        }
                    }
                    float* y = ytile + oc * plane;
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        float y0, y1;
                        if constexpr (S == 1) {
                            y0 = __builtin_fmaf(0.5f, s[i][1] + s[i][2], s[i][0]);
                            y1 = __builtin_fmaf(0.5f, s[i][1] - s[i][2], -s[i][3]);
                        } else {
                            y0 = s[i][0] + s[i][1];
                            y1 = s[i][1] + s[i][2];
                        }
                        y0 += bias[o][r], y1 += bias[o][r];
                        again |= (__builtin_fabsf(y0) < __builtin_inff() ? 0u : 1u) << (16 * o + 4 * r + 2 * i);
                        again |= (__builtin_fabsf(y1) < __builtin_inff() ? 0u : 2u) << (16 * o + 4 * r + 2 * i);
                        y0 = conv_finished(fin, y0, res[o][r][i][0]), y1 = conv_finished(fin, y1, res[o][r][i][1]);
                        if constexpr (FAST) {
                            *reinterpret_cast<f2*>(y + i * p.OW) = f2{y0, y1};
                        } else if (oc < p.OC && (i == 0 || below)) {
                            y[i * p.OW] = y0;
                            if (right) y[i * p.OW + 1] = y1;
                        }
                    }
                }
        };
        typedef std::integral_constant<bool, true> yes;
        typedef std::integral_constant<bool, false> no;
        const bool fast = pairs && oc0 + 32 <= p.OC && (p.OH & 1) == 0;
        if (tile_ok) {
            if (fin.residual) fast ? outputs(yes{}, yes{}) : outputs(no{}, yes{});
            else fast ? outputs(yes{}, no{}) : outputs(no{}, no{});
        }
        if (__ballot(again != 0) == 0) return;

        // The wavefront's outputs once more as direct sums, nine products for an output and channel on the same MFMA with pixels and filters as they lie (a tap in the
        // padding multiplies a zero, as in the other forms: an infinite weight gives a NaN there). Those that were not finite take them. With every
        // image a NaN 32 x 64 x 56 x 56 takes 227 us, 32 x 256 x 14 x 14 246 (direct 67 and 91; a lane and output at a time 3300 and 3000).
        int poff[PX][PX], foff[2];
#pragma unroll
        for (int r = 0; r < PX; r++)
#pragma unroll
            for (int c = 0; c < PX; c++) {
                const int ih = place.ih0 + r, iw = place.iw0 + c;
                const bool in = tile_ok && ih >= 0 && ih < p.H && iw >= 0 && iw < p.W;
                poff[r][c] = in ? ((n - place.n0) * p.XC * p.H * p.W + (lk * p.H + ih) * p.W + iw + kEarly) * 4 : kNone;
            }
#pragma unroll
        for (int o = 0; o < 2; o++) foff[o] = oc0 + o * 16 + l16 < p.OC ? ((o * 16 + l16) * p.C + lk) * 36 : kNone;
        wf4 sums[2][2][2];       // [row][column][block of channels]
#pragma unroll
        for (int q = 0; q < 8; q++) sums[q >> 2][(q >> 1) & 1][q & 1] = wf4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int step = 0; step < 2 * chunks; step++) {
            float x[PX][PX], w[2][9];
#pragma unroll
            for (int t = 0; t < 9; t++)
#pragma unroll
                for (int o = 0; o < 2; o++) w[o][t] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(place.wbuf, foff[o], step * 144 + t * 4, 0));
#pragma unroll
            for (int r = 0; r < PX; r++)
#pragma unroll
                for (int c = 0; c < PX; c++) x[r][c] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(place.xbuf, poff[r][c], step * 16 * p.H * p.W, 0));
#pragma unroll
            for (int t = 0; t < 9; t++)
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    const int i = q >> 2, j = (q >> 1) & 1, o = q & 1;
                    sums[i][j][o] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[o][t], x[S * i + t / 3][S * j + t % 3], sums[i][j][o], 0, 0, 0);
                }
        }
#pragma unroll
        for (int o = 0; o < 2; o++)
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int oc = oc0 + o * 16 + 4 * lk + r, i = q >> 1, j = q & 1;
                    if (!((again >> (16 * o + 4 * r + q)) & 1) || oc >= p.OC || oh + i >= p.OH || ow + j >= p.OW) continue;
                    const long to = oc * plane + (long) i * p.OW + j;
                    ytile[to] = conv_finished(fin, sums[i][j][o][r] + bias[o][r], fin.residual ? rtile[to] : -0.f);
                }
    }
};

} // namespace docc_k

namespace docc_k {
// sums: null, or where the part blockIdx.y of the channels (of gridDim.y) leaves its sums as [part][N][OC][OH][OW]
template <int S, int LOADS>
__device__ __forceinline__ void conv_winograd(ConvParams p, ConvFinish fin, float* sums) {
    typedef ConvWinograd<S> K;
    constexpr int TILES = 16 * K::NW;
    __shared__ __attribute__((aligned(16))) float lds[K::LDS_FLOATS];
    const int ocb = (p.OC + 31) >> 5, id = xcd_contiguous(blockIdx.x, gridDim.x);
    const int oc0 = (id % ocb) * 32, tile0 = (id / ocb) * TILES;
    int first = 0, chunks = p.C / K::CI;
    if (sums) {
        first = (int) ((long) chunks * blockIdx.y / gridDim.y);
        chunks = (int) ((long) chunks * (blockIdx.y + 1) / gridDim.y) - first;
        p.Y = sums + (long) blockIdx.y * p.N * p.OC * p.OH * p.OW;
        p.bias = nullptr;
        fin = ConvFinish{nullptr, 0};
    }
    if constexpr (S == 1 && LOADS != kPixels) {
        // the last tile that reads the column before the first row of the tensor (row 0 of image 0 is among its rows), and the first
        // that reads columns behind its last row
        const int TH = (p.OH + 1) >> 1, TW = (p.OW + 1) >> 1;
        const int before = (p.pad_h >> 1) * TW, bottom = (p.H - 3 + p.pad_h) >> 1;
        const long behind = (long) (p.N - 1) * TH * TW + (long) (bottom > 0 ? bottom : 0) * TW + TW - 1;
        if (tile0 > before && tile0 + TILES <= behind) K::template run<LOADS>(p, fin, lds, tile0, oc0, first * K::CI, chunks);
        else K::template run<kPixels>(p, fin, lds, tile0, oc0, first * K::CI, chunks);
    } else {
        K::template run<LOADS>(p, fin, lds, tile0, oc0, first * K::CI, chunks);
    }
}
} // namespace docc_k

#define DOCC_CONV_WINOGRAD(NAME, S, LOADS)                                                                                                \
    extern "C" __global__ __launch_bounds__(256, 2) void NAME(docc_k::ConvParams p, docc_k::ConvFinish f, float* sums) {                  \
        docc_k::conv_winograd<S, docc_k::LOADS>(p, f, sums);                                                                              \
    }
DOCC_CONV_WINOGRAD(docc_conv2d_f32_winograd_pixels, 1, kPixels)
DOCC_CONV_WINOGRAD(docc_conv2d_f32_winograd_vector, 1, kVector)
DOCC_CONV_WINOGRAD(docc_conv2d_f32_winograd_vector_odd, 1, kVectorOdd)
DOCC_CONV_WINOGRAD(docc_conv2d_f32_winograd_s2_vector, 2, kVector)
DOCC_CONV_WINOGRAD(docc_conv2d_f32_winograd_s2_pairs, 2, kPairs)
