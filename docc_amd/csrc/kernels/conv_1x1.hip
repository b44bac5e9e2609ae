// ml::Conv, 2-d NCHW fp32, 1x1 filters, with steps as the projection beside a block that halves the image has them: Y[oc, p] = sum_c W[oc, c] X[c, p'].
//
// Bound by little: 32 x 128 x 28 x 28 -> 256 with steps of two is 2.7 us of the fp32 matrix pipe and 4 us of memory (every line of X is touched, 12.8 MB,
// and 6.4 MB written). The strips of the LDS-halo kernel take the lines through LDS for a single use each: 19 us there, 13 us here. A wave takes 64 output
// channels x 16 pixels, lane l holding pixel l % 16 and the channels 4 (l / 16) .. + 3 of a step of sixteen: four loads of X that are the MFMAs' operands as they
// come. The filters of 32 channels at a time go through LDS for the four waves of a work-group (read from memory by each wave, rows of 512 bytes met
// in a few sets of the L1: 18 us), both two chunks ahead.
#include "elementwise_ops.h"
#include "conv_params.h"
#include <type_traits>

namespace docc_k {

__device__ __forceinline__ void conv1x1(const ConvParams& p, const ConvFinish& fin) {
    typedef float v4 __attribute__((ext_vector_type(4)));
    constexpr int ROW = 36, STAGE = 64 * ROW;      // floats: rows of 32 channels, four further apart (eight lanes read eight rows)
    __shared__ __attribute__((aligned(16))) float lds[3 * STAGE];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, lk = lane >> 4;
    const int plane = p.OH * p.OW, pixels = p.N * plane, ocb = (p.OC + 63) >> 6;
    const int id = xcd_contiguous(blockIdx.x, gridDim.x);
    const int oc0 = (id % ocb) * 64, pixel0 = (id / ocb) * 64;
    const int q = pixel0 + wave * 16 + l16;
    const bool ok = q < pixels;
    const int n0 = pixel0 / plane, n = (ok ? q : pixel0) / plane, at = (ok ? q : pixel0) % plane;
    const int ih = at / p.OW * p.stride_h - p.pad_h, iw = at % p.OW * p.stride_w - p.pad_w;
    const int HW4 = p.H * p.W * 4;

    constexpr int kNone = (int) 0x80000000;      // beyond the end of a buffer: the load gives 0
    const long left = (long) (p.N - n0) * p.C * HW4, wleft = (long) (p.OC - oc0) * p.C * 4;
    const auto xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.X) + (long) n0 * p.C * p.H * p.W, 0, (int) (left < 0x7fffffffL ? left : 0x7fffffffL), 0x00020000);
    const auto wbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.Wt) + (long) oc0 * p.C, 0, (int) (wleft < 0x7fffffffL ? wleft : 0x7fffffffL), 0x00020000);
    const bool in = ok && ih >= 0 && ih < p.H && iw >= 0 && iw < p.W;
    // this lane's pixel in the chunks of 32 channels, two steps of sixteen each; in the last chunk steps behind the last channel load nothing
    const int chunks = (p.C + 31) >> 5, last = chunks - 1;
    const int xoff = in ? ((n - n0) * p.C + 4 * lk) * HW4 + (ih * p.W + iw) * 4 : kNone;
    int xlast[2], woff[2], wlast[2];
    float* wdst[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        xlast[h] = last * 32 + h * 16 + 4 * lk < p.C ? xoff : kNone;
        // the vector of the filters this thread moves: 64 rows of eight
        const int row = (tid >> 3) + h * 32, c = (tid & 7) * 4;
        woff[h] = oc0 + row < p.OC ? (row * p.C + c) * 4 : kNone;
        wlast[h] = last * 32 + c < p.C ? woff[h] : kNone;
        wdst[h] = lds + row * ROW + c;
    }
    float b[3][2][4];
    v4 w[2];
    auto wload = [&](int chunk) {
        const int c = chunk < last ? chunk : last;          // (the last one once more)
#pragma unroll
        for (int h = 0; h < 2; h++) w[h] = __builtin_bit_cast(v4, __builtin_amdgcn_raw_buffer_load_b128(wbuf, c == last ? wlast[h] : woff[h], c * 128, 0));
    };
    auto wstore = [&](int buf) {
#pragma unroll
        for (int h = 0; h < 2; h++) *reinterpret_cast<v4*>(wdst[h] + buf * STAGE) = w[h];
    };
    auto xload = [&](int chunk, int to) {
        const int c = chunk < last ? chunk : last;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int off = c == last ? xlast[h] : xoff;
#pragma unroll
            for (int e = 0; e < 4; e++) b[to][h][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xbuf, off, (c * 32 + h * 16 + e) * HW4, 0));
        }
    };
    // the sums of a chunk are added up apart: 32 + C / 32 roundings in a chain instead of C (C = 288: 1.0e-7 off in the 2-norm, 2.5e-7 in one chain)
    v4 total[4];
#pragma unroll
    for (int o = 0; o < 4; o++) total[o] = v4{0.f, 0.f, 0.f, 0.f};
    wload(0);
    xload(0, 0);
    xload(1, 1);
    wstore(0);
    wload(1);
    __syncthreads();
    auto step = [&](int chunk, auto k_c) {
        constexpr int k = decltype(k_c)::value;
        wstore((k + 1) % 3);                                // last read two barriers ago
        wload(chunk + 2);
        xload(chunk + 2, (k + 2) % 3);
        __builtin_amdgcn_sched_barrier(0);
        v4 acc[4];
#pragma unroll
        for (int o = 0; o < 4; o++) acc[o] = v4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int h = 0; h < 2; h++) {
            v4 a[4];
#pragma unroll
            for (int o = 0; o < 4; o++) a[o] = *reinterpret_cast<const v4*>(lds + k * STAGE + (o * 16 + l16) * ROW + h * 16 + 4 * lk);
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int o = 0; o < 4; o++) acc[o] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[o][e], b[k][h][e], acc[o], 0, 0, 0);
        }
#pragma unroll
        for (int o = 0; o < 4; o++) total[o] += acc[o];
        __syncthreads();
    };
    int c = 0;
    for (; c + 2 < chunks; c += 3) {
        step(c, std::integral_constant<int, 0>{});
        step(c + 1, std::integral_constant<int, 1>{});
        step(c + 2, std::integral_constant<int, 2>{});
    }
    if (c < chunks) step(c, std::integral_constant<int, 0>{});
    if (c + 1 < chunks) step(c + 1, std::integral_constant<int, 1>{});

    if (!ok) return;
    const long to = (long) n * p.OC * plane + at;
#pragma unroll
    for (int o = 0; o < 4; o++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int oc = oc0 + o * 16 + 4 * lk + r;
            if (oc >= p.OC) continue;
            const long e = to + (long) oc * plane;
            p.Y[e] = conv_finished(fin, total[o][r] + (p.bias ? p.bias[oc] : -0.f), fin.residual ? fin.residual[e] : -0.f);
        }
}

} // namespace docc_k

extern "C" __global__ __launch_bounds__(256) void docc_conv2d_f32_1x1(docc_k::ConvParams p, docc_k::ConvFinish f) { docc_k::conv1x1(p, f); }
