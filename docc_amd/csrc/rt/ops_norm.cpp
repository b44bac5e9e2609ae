// Launcher of the layer normalisation kernels (see include/docc_rocm_ops.h, csrc/kernels/layernorm.hip).
#include <cstdio>
#include <cstdlib>

#include "docc_rocm_ops.h"
#include "rt_state.h"

using namespace docc::rt::rocm;

extern "C" int docc_rocm_layer_norm(docc_rocm_stream_t stream, int type, int64_t rows, int64_t cols, float eps, const void* X, const void* weight,
                                    const void* bias, void* Y) {
    if (type != DOCC_ROCM_TYPE_F32 && type != DOCC_ROCM_TYPE_BF16) return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "layer_norm: float32 or bf16 tensors");
    if (rows < 0 || cols < 0) return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "layer_norm: negative dimension");
    if (rows == 0 || cols == 0) return 0;
    if (!X || !Y) return fail(DOCC_ROCM_ERR_INVALID_ARGUMENT, "layer_norm: null pointer");
    if (int rc = ensure_device()) return rc;
    int cus = compute_units();
    if (cus <= 0) cus = 256;
    const bool bf16 = type == DOCC_ROCM_TYPE_BF16;
    const int full = bf16 ? 8 : 4;
    const bool vec = cols % full == 0 && ((uintptr_t) X | (uintptr_t) weight | (uintptr_t) bias | (uintptr_t) Y) % 16 == 0;
    const int64_t lane = vec ? full : 1;   // elements of a lane's access
    // vectors a lane holds with `lanes` of them on a row: the smallest built count that covers the row, 0 if none does
    auto held = [&](int64_t lanes) -> int {
        const int64_t n = (cols + lanes * lane - 1) / (lanes * lane);
        if (!vec) return n <= 4 ? 4 : lanes == 256 && n <= 16 ? 16 : 0;
        return n <= 1 ? 1 : n <= 2 ? 2 : n <= 4 ? 4 : !bf16 && lanes == 256 && n <= 8 ? 8 : 0;
    };
    // a wavefront a row where that gives every CU its four rows, or where a row is one access of 64 lanes
    const int w = held(64), b = held(256);
    const bool wave = w != 0 && (rows >= 4 * (int64_t) cus || cols <= 64 * lane);
    // short rows: a power of two of lanes, at most 32, with a vector or four elements each
    const int64_t wanted = (cols + (vec ? full : 4) - 1) / (vec ? full : 4);
    int64_t sub = 1;
    while (sub < wanted && sub < 64) sub *= 2;
    const bool part = sub <= 32;
    char name[64];
    const bool one = !part && !wave && !b;   // a work-group of 1024 a row
    if (part) std::snprintf(name, sizeof(name), "docc_layernorm_%s_%c_p%d", bf16 ? "bf16" : "f32", vec ? 'v' : 's', (int) sub);
    else if (one) std::snprintf(name, sizeof(name), "docc_layernorm_%s_long", bf16 ? "bf16" : "f32");
    else std::snprintf(name, sizeof(name), "docc_layernorm_%s_%c_%c%d", bf16 ? "bf16" : "f32", vec ? 'v' : 's', wave ? 'w' : 'b', wave ? w : b);
    if (one) {
        // Rows in slices: three launches, from 16384 columns on faster than a work-group a row whatever their number (fp32, rows x columns, a
        // work-group a row / slices: 4 x 12000 9.7 / 11.5 us, 4 x 20000 14.6 / 11.8, 1 x 2^20 1241 / 11, 1024 x 20000 65 / 53, 256 x
        // 200704 320 / 146); without whole vectors up to a row a CU (256 x 33333 45 / 42, 512 x 33333 54 / 77).
        // DOCC_ROCM_LAYERNORM=slices|rows takes one or the other (tests, tuning).
        const char* force = std::getenv("DOCC_ROCM_LAYERNORM");
        const bool pays = cols > 16384 && (vec || rows <= cus);
        int64_t slices = rows < 4 * (int64_t) cus ? 4 * (int64_t) cus / rows : 1;
        if (slices > 256) slices = 256;
        if (slices > cols / 2048) slices = cols / 2048 > 1 ? cols / 2048 : 1;
        const int64_t chunk = ((cols + slices - 1) / slices + lane - 1) / lane * lane;
        slices = (cols + chunk - 1) / chunk;
        hipStream_t s = (hipStream_t) stream;
        PartialsLease lease;
        if ((force ? force[0] == 's' : pays) && rows <= 65535 && 2 * rows * slices * (int64_t) sizeof(float) <= (int64_t) kPartialsBytes &&
            (!foreign_capture(s) || partials_held(s)) && partials_for(s, &lease) == 0) {
            float *sums = (float*) lease.ptr, *squares = sums + rows * slices;
            auto step = [&](const char* what, auto... args) {
                std::snprintf(name, sizeof(name), "docc_layernorm_%s_%c_slice_%s", bf16 ? "bf16" : "f32", vec ? 'v' : 's', what);
                return launch(name, (uint32_t) slices, (uint32_t) rows, 1, 256, 0, s, (long) cols, (long) chunk, args...);
            };
            int rc = step("sum", X, sums);
            if (!rc) rc = step("squares", X, (const float*) sums, squares);
            if (!rc) rc = step("apply", eps, X, (const float*) sums, (const float*) squares, weight, bias, Y);
            return rc;
        }
    }
    // a launch holds fewer than 2^32 threads: more rows than that takes go in several
    const int64_t threads = one ? 1024 : 256, per_group = part ? 256 / sub : wave ? 4 : 1, most = ((int64_t(1) << 32) / threads - 1) * per_group;
    const int64_t row_bytes = cols * (bf16 ? 2 : 4);
    for (int64_t r0 = 0; r0 < rows; r0 += most) {
        const int64_t n = rows - r0 < most ? rows - r0 : most;
        const int rc = launch(name, (uint32_t) ((n + per_group - 1) / per_group), 1, 1, (uint32_t) threads, 0, (hipStream_t) stream, (long) n, (long) cols,
                              eps, (const void*) ((const char*) X + r0 * row_bytes), weight, bias, (void*) ((char*) Y + r0 * row_bytes));
        if (rc) return rc;
    }
    return 0;
}
