"""What the launchers ask of the HIP runtime, on the CPU: the library runs in a process of its own on a recorder of the HIP host API
(hip_recorder.c), which writes down allocations, events, waits and launches. No kernel runs, so what is checked is the order of
the calls: whose memory a launch uses, and what stands between a block's release and its next owner."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
PRELUDE = f"""
import ctypes, sys
sys.path.insert(0, {str(HERE.parent)!r})
recorder = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
recorder.recorder_take.restype = ctypes.c_char_p
recorder.recorder_capture.argtypes = [ctypes.c_void_p]
recorder.recorder_no_memory_from.argtypes = [ctypes.c_size_t]
from docc_amd import runtime as rt
rt.init(0)
A, B, C, D = 0x10000000, 0x20000000, 0x30000000, 0x40000000     # operands: numbers, nothing reads them
def take():
    return recorder.recorder_take().decode().splitlines()
"""


@pytest.fixture(scope="module")
def recorded(tmp_path_factory):
    """Runs a script behind PRELUDE; what it prints, as lines."""
    lib = tmp_path_factory.mktemp("recorder") / "librecorder.so"
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-I", f"{rocm}/include", str(HERE / "hip_recorder.c"), "-o", str(lib)], check=True)

    def run(script, **env):
        clean = {k: v for k, v in os.environ.items() if not k.startswith("DOCC_ROCM_")}
        done = subprocess.run([sys.executable, "-c", PRELUDE + script, str(lib)], capture_output=True, text=True, env={**clean, **env}, timeout=60)
        assert done.returncode == 0, done.stderr
        return done.stdout.splitlines()

    return run


# a packed product; K in parts whose sums exceed the stream's buffer; few rows in parts of the same size; a few columns held row by row
GEMMS = {"packed": "rt.bf16gemm_f32(4096, 4096, 4097, 1.0, A, 4097, B, 4096, 0.0, C, 4096, stream=s)",
         "parts": "rt.sgemm(512, 1024, 8192, 1.0, A, 8192, B, 1024, 0.0, C, 1024, stream=s)",
         "few rows": "rt.sgemm(32, 16384, 16384, 1.0, A, 16384, B, 16384, 0.0, C, 16384, stream=s)",
         "few columns": "rt.sgemm(4096, 9, 4096, 1.0, A, 4096, B, 9, 0.0, C, 9, stream=s)"}


@pytest.mark.parametrize("what", list(GEMMS))
def test_a_product_takes_no_block_where_none_can_be_kept_for_it(recorded, what):
    script = f"""
def gemm(s): {GEMMS[what]}
s = rt.stream_create()
gemm(s)
usual = take()
assert any(l.startswith("malloc") and l != "malloc 8388608" for l in usual), usual      # (that size: the stream's own buffer, kept)
rt.pool_trim()
take()
# a graph that another library records would go on writing to a block that has been given back
recorder.recorder_capture(s)
gemm(s)
got = take()
assert got and all(l.startswith("launch") for l in got), got
recorder.recorder_capture(None)
# without memory the product runs on what it has, and leaves no error behind for other users of the HIP runtime
recorder.recorder_no_memory_from(1)
gemm(s)
got = take()
assert all(l.startswith("launch") or l.endswith("refused") for l in got) and got[-1].startswith("launch"), got
assert recorder.hipGetLastError() == 0
"""
    recorded(script, **({"DOCC_ROCM_GEMM_SPLITK": "16"} if what == "few rows" else {}))


def test_a_layer_that_needs_a_block_is_refused_in_a_foreign_capture(recorded):
    recorded("""
s = rt.stream_create()
def linear(n): rt.call("docc_rocm_linear", s, 2, 111, 112, 256, n, 64, 1.0, A, 64, B, 64, None, 2, 16, None, 2, 0, D, 2)
linear(100)
assert any(l.startswith("malloc") for l in take())
recorder.recorder_capture(s)
linear(128)                       # the chain is in the product's store
assert [l.split()[0] for l in take()] == ["launch"]
try:
    linear(100)                   # no whole vectors: through memory
    assert False
except rt.RocmRuntimeError as e:
    assert "capture" in str(e), e
assert take() == []
""")


def test_attention_and_convolution_run_whole_in_a_foreign_capture_or_without_memory(recorded):
    recorded("""
s = rt.stream_create()
def attention(): rt.attention_bf16(1, 4, 1, 32768, 128, 0.1, A, B, C, D, stream=s)
W = 0x50000000
def conv(): rt.conv2d_f32(1, 256, 14, 14, 256, 3, 3, (1, 1), (1, 1), (1, 1), A, B, C, D, stream=s)
for call in (attention, conv):
    call()
    usual = take()
    assert any(l.startswith("malloc") for l in usual) and len([l for l in usual if l.startswith("launch")]) == 2, usual
    rt.pool_trim()
    take()
    recorder.recorder_capture(s)
    call()
    got = take()
    assert [l.split()[0] for l in got] == ["launch"], got
    recorder.recorder_capture(None)
    recorder.recorder_no_memory_from(1)
    call()
    got = take()
    assert got[0].endswith("refused") and [l.split()[0] for l in got if not l.endswith("refused")] == ["launch"], got
    assert recorder.hipGetLastError() == 0
    recorder.recorder_no_memory_from(ctypes.c_size_t(-1))
# with a workspace a convolution that cannot be cut takes the form that was the fastest before
size = (8, 256, 14, 14, 256, 3, 3, (1, 1), (1, 1), (1, 1))
need = rt.conv2d_f32_workspace_bytes(*size)
assert need > 0
rt.conv2d_f32_ws(*size, A, B, C, D, W, need, stream=s)
assert "_parts" in " ".join(take())
recorder.recorder_capture(s)
rt.conv2d_f32_ws(*size, A, B, C, D, W, need, stream=s)
got = " ".join(take())
assert "im2col" in got and "sgemm" in got and "malloc" not in got, got
""")


@pytest.mark.parametrize("rows,cols,launches", [(2 ** 24 + 5, 2000, 2), (2 ** 26 + 1, 256, 2), (2 ** 32, 4, 2), (2 ** 22, 16384, 2), (2 ** 24 - 1, 2000, 1)])
def test_layer_norm_of_more_rows_than_a_launch_holds(recorded, rows, cols, launches):
    # 2^32 threads are one too many for a launch (the recorder refuses them as the device does)
    got = recorded(f"""
rt.call("docc_rocm_layer_norm", 0, 2, {rows}, {cols}, 1e-5, A, None, None, B)
print("\\n".join(take()))
""")
    assert len(got) == launches and all(l.startswith("launch docc_layernorm_f32") for l in got)


# a product with fewer tiles than CUs (a dozen numbers of parts on four tiles each), and attention: once for the entry point, once for the
# planning, and once a launch, an allocation and a release
@pytest.mark.parametrize("call,most", [("rt.bf16gemm_f32(512, 512, 4096, 1.0, A, 4096, B, 512, 0.0, C, 512)", 8),
                                       ("rt.attention_bf16(4, 16, 64, 64, 64, 0.1, A, B, C, D)", 3)])
def test_a_call_asks_for_the_device_a_few_times_however_many_forms_it_weighs(recorded, call, most):
    got = recorded(f"""
for _ in range(2):
    recorder.recorder_device_queries()
    {call}
print(recorder.recorder_device_queries())
""")
    assert int(got[0]) <= most


@pytest.mark.parametrize("form,channels,parts", [("t4-parts2", 32, 2), ("t2-parts2", 32, 2), ("t4m-parts3", 72, 3), ("t2m-parts4", 72, 4), ("t4-parts2", 24, 0)])
def test_convolutions_in_a_given_form_and_number_of_parts(recorded, form, channels, parts):
    got = recorded(f"""
rt.conv2d_f32(5, {channels}, 9, 7, 70, 3, 3, (1, 1), (1, 1), (1, 1), A, B, C, D)
print("\\n".join(l for l in take() if l.startswith("launch")))
""", DOCC_ROCM_CONV="halo-" + form)
    assert len(got) == (2 if parts else 1)          # fewer than four chunks of channels are not cut
    if parts:
        assert f"_{form.split('-')[0]}_parts " in got[0] and f",2,{parts} " in got[0] and "add_parts" in got[1]


# what the planner takes by itself: the shapes of tests/test_gpu_conv_parts.py are products of the cut form, in the form that is chosen and among the direct ones
def test_few_images_of_many_channels_are_cut(recorded):
    from test_gpu_conv_parts import test_channels_in_parts as cases
    rows = next(m for m in cases.pytestmark if m.name == "parametrize").args[1]
    for N, C, OC, H, W, k, stride, pad, _ in rows:
        got = recorded(f"""
rt.conv2d_f32({N}, {C}, {H}, {W}, {OC}, {k}, {k}, ({stride}, {stride}), ({pad}, {pad}), (1, 1), A, B, C, D)
print("\\n".join(l for l in take() if l.startswith("launch")))
""")
        assert ("_parts" in " ".join(got)) == (C > 16), (N, C, got)
        got = recorded(f"""
rt.conv2d_f32({N}, {C}, {H}, {W}, {OC}, {k}, {k}, ({stride}, {stride}), ({pad}, {pad}), (1, 1), A, B, C, D)
print("\\n".join(l for l in take() if l.startswith("launch")))
""", DOCC_ROCM_CONV="direct")
        first = got[0].split()
        assert first[1].startswith("docc_conv2d_f32_halo_") and first[1].endswith("_parts") == (C > 16) and (int(first[2].split(",")[2]) > 1) == (C > 16), (N, C, got)


# ... and the layers of tests/test_gpu_conv.py that are named for their columns and GEMM take them when asked to, with a workspace
def test_layers_as_columns_and_gemm(recorded):
    from test_gpu_conv import GEMM_LAYERS
    for N, C, H, W, OC, KH, KW, stride, pad, dil, _ in GEMM_LAYERS:
        for force, first in (("gemm", "docc_conv2d_im2col_f32" if KH == 3 else "gemm"), ("gather", "docc_conv2d_f32"), ("halo-t2", "docc_conv2d_f32_halo_")):
            got = recorded(f"""
size = ({N}, {C}, {H}, {W}, {OC}, {KH}, {KW}, {stride}, {pad}, {dil})
need = rt.conv2d_f32_workspace_bytes(*size)
rt.conv2d_f32_ws(*size, A, B, C, D, 0x50000000 if need else 0, need)
print("\\n".join(l for l in take() if l.startswith("launch")))
""", DOCC_ROCM_CONV=force)
            assert first in " ".join(got) and "winograd" not in " ".join(got), (N, C, force, got)


# the products of tests/test_gpu_gemm.py with one to eight rows or columns on the matrix-vector kernels, with the switch that its second run sets
def test_few_rows_or_columns_without_the_kernels_that_cut_k_between_wavefronts(recorded):
    from test_gpu_gemm import GEMV_CASES
    for m, n, k, ta, tb in GEMV_CASES:
        got = recorded(f"""
rt.sgemm({m}, {n}, {k}, 1.0, A, {m if ta == 112 else k}, B, {k if tb == 112 else n}, 0.0, C, {n}, trans_a={ta}, trans_b={tb})
print("\\n".join(l for l in take() if l.startswith("launch")))
""", DOCC_ROCM_GEMM_WAVES="0")
        tiles = (m, n, ta, tb) in ((8, 4200, 111, 111), (4100, 8, 112, 111))       # (eight vectors along the other operand's rows: there the tiles' margins are tried)
        assert "waves" not in " ".join(got) and any("gemv" in l for l in got) != tiles, (m, n, k, got)


def test_the_release_of_a_block_of_the_null_stream_is_recorded_when_somebody_else_takes_it(recorded):
    recorded("""
n, b = 1 << 20, rt.stream_create()
p = rt.malloc_async(n)
take()
rt.free_async(p)
assert rt.malloc_async(n) == p and take() == []                     # the same stream: nothing recorded, nothing waited for
rt.free_async(p)
assert rt.malloc_async(n, b) == p
assert take() == ["event 1", "record 1 on (nil)", f"{b:#x} waits for 1"]
rt.free_async(p, b)
assert take() == ["record 1 on " + f"{b:#x}"]                        # any other stream may be gone by then: at once
assert rt.malloc(n) == p
assert take() == ["host waits for 1"]
rt.free_async(p)
assert take() == []
assert rt.malloc(n) == p
assert take() == ["record 1 on (nil)", "host waits for 1"]           # the event came along
rt.set_default_stream(b)
rt.free_async(p)                                                      # the null stream stands for b here
assert take() == ["record 1 on " + f"{b:#x}"]
""")


# bf16 products on which one tile was measured to be the fastest by a tenth or more, and one with an epilogue that parts of K do not pay for
@pytest.mark.parametrize("m,n,k,ta,tb,epilogue,kernel", [(1509, 2816, 1032, 0, 0, 0, "128x128x32s4_nn"), (2944, 2912, 688, 0, 0, 1, "128x128x32s4_nn_e"),
                                                         (3064, 1408, 3552, 0, 0, 0, "128x128x32s4_nn"), (4096, 4096, 4096, 0, 0, 0, "256x256x32q4_nn"),
                                                         (4096, 2048, 8192, 0, 1, 0, "128x256x64s3_nt"), (2048, 2048, 2048, 0, 0, 0, "128x128x64s4_nn"),
                                                         (5352, 3072, 96, 0, 0, 1, "128x128x32s4_nn_e"), (64, 192, 1093, 1, 0, 1, "128x128x32s4_tn_e"),
                                                         (3, 192, 768, 0, 1, 0, "128x128x32s4_nt"), (512, 256, 2048, 0, 1, 1, "128x128x32s4_nt_e")])
def test_tiles_of_bf16_products(recorded, m, n, k, ta, tb, epilogue, kernel):
    got = recorded(f"""
rt.call("docc_rocm_bf16gemm_f32_epilogue", 0, {111 + ta}, {111 + tb}, {m}, {n}, {k}, 1.0, A, {m if ta else k}, B, {k if tb else n}, 0.0, C, {n}, D if {epilogue} else None,
        2 if {epilogue} else -1)
print("\\n".join(l for l in take() if l.startswith("launch")))
""")
    assert len(got) == 1 and got[0].split()[1] == "docc_bgemma_" + kernel, got


# long rows go in slices, several work-groups a row where there are few of them; not in a capture on a stream that has no buffer for their sums
@pytest.mark.parametrize("rows,cols,groups", [(1, 2 ** 20, "256,1,1"), (32, 200704, "32,32,1"), (2000, 20000, "1,2000,1"), (3, 33333, "16,3,1"), (2, 16384, None),
                                              (300, 33333, None), (70000, 20000, None)])
def test_layer_norm_of_long_rows(recorded, rows, cols, groups):
    recorded(f"""
s = rt.stream_create()
def norm(): rt.call("docc_rocm_layer_norm", s, 2, {rows}, {cols}, 1e-5, A, None, None, B)
def launches(): return [l for l in take() if l.startswith("launch")]
recorder.recorder_capture(s)
norm()
assert all("_f32_long" in l for l in launches())
recorder.recorder_capture(None)
norm()
got = launches()
if {groups!r} is None:
    assert all("_f32_long" in l for l in got), got
else:
    assert [l.split()[1].split("_slice_")[1] for l in got] == ["sum", "squares", "apply"] and all(" {groups} x 256 " in l for l in got), got
    recorder.recorder_capture(s)
    norm()
    assert launches() == got
""")


@pytest.mark.parametrize("cols,form", [(4, "v_p1"), (8, "v_p2"), (24, "v_p8"), (128, "v_p32"), (132, "v_w1"), (3, "s_p1"), (5, "s_p2"), (30, "s_p8"), (127, "s_p32"), (129, "s_w4")])
def test_layer_norm_of_short_rows(recorded, cols, form):
    got = recorded(f"""
rt.call("docc_rocm_layer_norm", 0, 2, 100000, {cols}, 1e-5, A, None, None, B)
print(take()[0])
""")
    assert got[0].split()[1] == "docc_layernorm_f32_" + form
    if "p" in form:
        per_group = 256 // int(form.split("p")[1])
        assert f" {-(-100000 // per_group)},1,1 x 256 " in got[0]


# k off the vectors: packed where that was measured to be faster, plain where the packed product's tiles end in a nearly empty round
@pytest.mark.parametrize("m,n,k,packed", [(2048, 2048, 2047, True), (300, 300, 8001, True), (5120, 2304, 1391, False), (3000, 500, 300, False)])
def test_operands_off_the_vectors_are_packed_where_it_pays(recorded, m, n, k, packed):
    got = recorded(f"""
rt.sgemm({m}, {n}, {k}, 1.0, A, {k}, B, {k}, 0.0, C, {n}, trans_b=rt.TRANS)
print("\\n".join(l for l in take() if l.startswith("launch")))
""")
    assert ("docc_gemm_pack_b4" in got[0]) == packed, got


# the shapes of tests/test_gpu_gemm_pack.py whose K is to be cut into parts of different lengths are cut so, with the switch that its second run sets
@pytest.mark.parametrize("kind", ["dgemm", "sgemm", "bf16gemm_f32"])
def test_k_is_cut_into_parts_of_different_lengths(recorded, kind):
    from test_gpu_gemm_pack import test_parts_of_different_lengths as cases
    shapes = next(m for m in cases.pytestmark if m.name == "parametrize" and "m,n,k" in m.args[0]).args[1]
    for m, n, k in shapes:
        got = recorded(f"""
rt.{kind}({m}, {n}, {k}, 1.0, A, {k}, B, {k}, 0.0, C, {n}, trans_b=rt.TRANS)
print("\\n".join(l for l in take() if l.startswith("launch")))
""", DOCC_ROCM_GEMM_WAVES="0")
        parts = int(got[0].split()[2].split(",")[1])
        part = ((k + parts - 1) // parts + 63) // 64 * 64
        if (kind, m) == ("bf16gemm_f32", 16):
            assert len(got) == 1            # one tile of 128 x 128, which parts of 256 k do not pay for
        else:
            assert parts > 1 and "splitk_combine" in got[1] and k % part, (m, n, k, got)


# a norm and a layer in one launch, but in two where that one would read what it stores, or what it does not store
def test_a_norm_and_a_layer_on_operands_that_overlap(recorded):
    recorded("""
m, n, k = 8, 512, 256                                    # rows of X: 1024 bytes, of Y: 2048
G, H, W, BIAS, S = (0x50000000 + i * 0x1000000 for i in range(5))
def launches(X=A, weight=G, shift=H, w=W, bias=BIAS, residual=C, scratch=S, y=D, type=2, m=m, n=n):
    rt.call("docc_rocm_norm_linear", 0, type, m, n, k, 1e-5, X, weight, shift, 1.0, w, k, bias, type, -1, residual, type, 0, scratch, y, type)
    return len([l for l in take() if l.startswith("launch")])
rows, out = m * k * 4, m * n * 4
assert launches() == launches(type=1) == launches(residual=D) == launches(scratch=A) == 1
assert launches(X=A, residual=A, y=A, n=k) == 2          # in place
assert launches(X=A, residual=A, y=A, n=k, type=1) == 2
assert launches(X=D + out) == launches(X=D - rows) == 1  # side by side
assert launches(X=D + out - 16) == launches(X=D - rows + 16) == 2
assert launches(weight=D) == launches(weight=D + out - 16) == launches(weight=D - k * 4 + 16) == launches(shift=D + 16) == 2
assert launches(weight=D + out) == launches(shift=D - k * 4) == 1
assert launches(residual=S) == launches(residual=S + rows - 16) == launches(residual=S - out + 16) == launches(w=S) == launches(bias=S + 16) == 2
assert launches(residual=S + rows) == launches(w=S + rows) == launches(bias=S - n * 4) == 1
""")


# a vector of a row of odd length reaches into the next row, and that of an image one pixel wide a row further: it goes pixel by pixel
@pytest.mark.parametrize("height,width,form", [(258, 1, "pixels"), (7, 1, "pixels"), (258, 3, "vector_odd"), (258, 2, "vector")])
def test_loads_of_narrow_images_in_winograds_form(recorded, height, width, form):
    got = recorded(f"""
rt.conv2d_f32(1, 64, {height}, {width}, 64, 3, 3, (1, 1), (1, 1), (1, 1), A, B, C, D)
print("\\n".join(l for l in take() if l.startswith("launch")))
""", DOCC_ROCM_CONV="winograd")
    assert got[0].split()[1] == "docc_conv2d_f32_winograd_" + form


# an error's code is HIP's, and that of a copy with invalid arguments is 1: after it some rows have been written, so the call is not done again
@pytest.mark.parametrize("failing", [0, 1, 4, 15])
@pytest.mark.parametrize("pinned", [False, True])
def test_a_copy_that_fails_among_chunks_fails_the_call(recorded, failing, pinned):
    recorded(f"""
import numpy as np
shape = (4096, 2048)                                      # 32 MB, eight chunks
y = rt.result_array(shape, np.float32)
x = rt.result_array(shape, np.float32) if {pinned} else np.empty(shape, np.float32)
def softmax(x): rt.call("docc_rocm_softmax_host", 0, 32, *shape, 1, x.ctypes.data, y.ctypes.data)
softmax(x)
whole = [l for l in take() if l.startswith("copy")]
assert len(whole) == 16 and all(" 4194304 " in l for l in whole), whole
for source in (x, y):                                     # y: in place
    recorder.recorder_fail_copy({failing})
    try:
        softmax(source)
        assert False
    except rt.RocmRuntimeError as e:
        assert "hipMemcpyAsync" in str(e), e
    got = [l for l in take() if l.startswith("copy")]
    assert len(got) == {failing} + 1 and got[-1].endswith("failed"), got
# an upload through pinned buffers too
if not {pinned}:
    recorder.recorder_fail_copy(1)
    try:
        rt.call("docc_rocm_memcpy_h2d_async", A, x.ctypes.data, x.nbytes, 0)
        assert False
    except rt.RocmRuntimeError as e:
        assert "hipMemcpyAsync" in str(e), e
    assert len([l for l in take() if l.startswith("copy")]) == 2
# where nothing can be set up the array goes as a whole
recorder.recorder_fail_copy(-1)
recorder.recorder_no_memory_from(1 << 20)
rt.pool_trim()
take()
try:
    softmax(x)
    assert False
except rt.RocmRuntimeError as e:
    assert "emory" in str(e), e
assert not [l for l in take() if l.startswith("copy")]
""")


# Winograd's form from 32 channels on, and in parts where the direct sum would be in so many that the whole would be further off; not at all where the caller says so
@pytest.mark.parametrize("N,C,size,stride,parts", [(4, 8, 28, 1, 0), (64, 8, 56, 1, 0), (32, 16, 56, 1, 0), (8, 24, 28, 2, 0), (64, 32, 56, 1, 1), (12, 48, 27, 1, 3), (15, 48, 21, 1, 3),
                                                   (4, 32, 17, 2, 2), (32, 128, 28, 2, 1)])
def test_chains_of_sums_in_winograds_form(recorded, N, C, size, stride, parts):
    for choice in ("", "direct"):
        got = recorded(f"""
rt.conv2d_f32({N}, {C}, {size}, {size}, {C * stride}, 3, 3, ({stride}, {stride}), (1, 1), (1, 1), A, B, C, D)
print("\\n".join(l for l in take() if l.startswith("launch")))
""", **({"DOCC_ROCM_CONV": choice} if choice else {}))
        assert ("winograd" in got[0]) == (parts > 0 and not choice), got
        if "winograd" in got[0]:
            assert f",{parts},1 x" in got[0], got


# generated code asks for a column matrix where the call reads it, and a call that does not read one is the same without
@pytest.mark.parametrize("size", [(8, 256, 14, 14, 256, 1), (64, 256, 7, 7, 256, 2), (25, 416, 12, 12, 416, 1), (1, 256, 14, 14, 256, 1), (16, 40, 30, 30, 40, 1), (2, 64, 5, 500, 64, 1),
                                  (3, 20, 20, 20, 50, 1), (8, 100, 14, 14, 256, 1)])
def test_a_workspace_is_asked_for_where_it_is_read(recorded, size):
    recorded(f"""
N, C, H, W, OC, stride = {size}
size = (N, C, H, W, OC, 3, 3, stride, stride, 1, 1, 1, 1, 1, 1)
need = rt.lib().docc_rocm_conv2d_f32_pads_workspace_bytes(*size)
def names(workspace):
    rt.call("docc_rocm_conv2d_f32_pads", s, *size, A, B, C_, D, workspace, need if workspace else 0)
    return [l.split()[1] for l in take() if l.startswith("launch")]
C_, s = 0x60000000, 0
reads = rt.lib().docc_rocm_conv2d_f32_reads_workspace(s, *size, B)
assert need > 0 or not reads
assert reads == (need > 0 and "docc_conv2d_im2col_f32" in names(0x50000000))
if not reads: assert names(0x50000000 if need else None) == names(None)
# in another library's capture, where the channels cannot be cut
s = rt.stream_create()
recorder.recorder_capture(s)
reads = rt.lib().docc_rocm_conv2d_f32_reads_workspace(s, *size, B)
assert reads == (need > 0 and "docc_conv2d_im2col_f32" in names(0x50000000))
""")


def test_a_layer_in_winograds_form_asks_for_no_column_matrix(recorded):
    got = recorded("""
import random, math
rng = random.Random(1)
asked = 0
for _ in range(300):
    N, C, size, stride = round(math.exp(rng.uniform(0, 4.1))), 16 * round(math.exp(rng.uniform(0.7, 3.4))), rng.randint(7, 64), rng.choice([1, 1, 2])
    shape = (N, C, size, size, C * stride, 3, 3, stride, stride, 1, 1, 1, 1, 1, 1)
    rt.call("docc_rocm_conv2d_f32_pads", 0, *shape, A, B, None, D, None, 0)
    if "winograd" in next(l for l in take() if l.startswith("launch")):
        asked += rt.lib().docc_rocm_conv2d_f32_reads_workspace(0, *shape, B)
print(asked)
""")
    assert int(got[0]) == 0


# K between the wavefronts of a work-group whether it is a multiple of their rounds or not; in fp64 not where rows off the lines of 128 bytes are read over and over
@pytest.mark.parametrize("kind,m,n,k,waves", [("s", 512, 512, 512, True), ("s", 512, 512, 576, True), ("s", 512, 512, 580, True), ("s", 204, 172, 100, True), ("s", 1402, 409, 32, False),
                                              ("d", 512, 512, 512, True), ("d", 512, 512, 514, True), ("d", 97, 744, 286, True), ("d", 285, 205, 56, False),
                                              ("d", 968, 183, 5886, False), ("d", 266, 1411, 3730, False), ("d", 1242, 251, 3584, False), ("d", 216, 906, 3844, True)])
def test_k_off_the_rounds_of_the_wavefronts(recorded, kind, m, n, k, waves):
    got = recorded(f"""
rt.{kind}gemm({m}, {n}, {k}, 1.0, A, {k}, B, {k}, 0.0, C, {n}, trans_b=rt.TRANS)
print("\\n".join(l for l in take() if l.startswith("launch")))
""")
    assert ("_waves_" in got[0]) == waves, got


# 1x1 layers: on the kernel that takes the pixels as they lie, but few channels on many work-groups on the strips, and without anything behind the product on the batched
# product, unless many work-groups share many output channels
@pytest.mark.parametrize("N,C,H,W,OC,stride,bias,kernel", [(32, 128, 28, 28, 256, 2, True, "f32_1x1"), (16, 128, 28, 28, 512, 1, True, "f32_1x1"), (49, 8, 32, 32, 133, 1, True, "halo"),
                                                           (59, 8, 60, 62, 24, 1, False, "halo"), (34, 12, 61, 52, 10, 1, True, "gather"), (5, 8, 34, 34, 296, 1, True, "f32_1x1"),
                                                           (56, 208, 64, 19, 192, 1, True, "f32_1x1"), (56, 208, 64, 19, 192, 1, False, "gemm"), (3, 232, 16, 16, 514, 1, False, "gemm"),
                                                           (3, 176, 34, 34, 1400, 1, False, "f32_1x1"), (3, 160, 21, 33, 83, 1, False, "f32_1x1")])
def test_kernels_of_1x1_layers(recorded, N, C, H, W, OC, stride, bias, kernel):
    got = recorded(f"""
rt.conv2d_f32({N}, {C}, {H}, {W}, {OC}, 1, 1, ({stride}, {stride}), (0, 0), (1, 1), A, B, C if {bias} else 0, D)
print("\\n".join(l for l in take() if l.startswith("launch")))
""")
    assert kernel in " ".join(got) and len(got) == 1, got
    if not bias:        # the sum with a tensor is a pass of its own behind the batched product too
        got = recorded(f"""
rt.call("docc_rocm_conv2d_f32_chain", 0, {N}, {C}, {H}, {W}, {OC}, 1, 1, {stride}, {stride}, 0, 0, 0, 0, 1, 1, 1, A, B, None, C, -1, D, None, 0)
print("\\n".join(l for l in take() if l.startswith("launch")))
""")
        assert ("f32_1x1" in got[0]) == (kernel != "halo") and len(got) == (2 if kernel == "halo" else 1), got


# layers in bf16: K between the wavefronts, but not where the rows of many tiles are read from beyond the caches, off the lines of 128 bytes above all
@pytest.mark.parametrize("m,n,k,waves", [(1024, 1024, 256, True), (162, 2208, 3096, True), (98, 6776, 1864, True), (596, 2664, 3880, False), (720, 2464, 4696, False), (146, 1952, 6488, False),
                                         (489, 3408, 4680, False), (124, 1936, 3848, True), (644, 5696, 4416, False), (302, 2704, 5504, True)])
def test_layers_with_long_rows(recorded, m, n, k, waves):
    got = recorded(f"""
rt.call("docc_rocm_linear", 0, 1, 111, 112, {m}, {n}, {k}, 1.0, A, {k}, B, {k}, C, 1, 2, None, 1, 0, D, 1)
print("\\n".join(l for l in take() if l.startswith("launch")))
""")
    assert ("_waves_" in got[0]) == waves, got
