"""Launches merged when host code is generated: what is emitted for a layer and for a layer norm spelled with tensor nodes, and what
keeps its separate launches."""
import json
import re

import pytest
import torch
import torch.nn.functional as F

import docc_amd.torch as docc_torch
from docc_amd.sdfg import Pointer, PrimitiveType, Scalar, StructuredSDFG, StructuredSDFGBuilder

F32, F64 = Pointer(Scalar(PrimitiveType.Float)), Pointer(Scalar(PrimitiveType.Double))


def calls(sdfg, folder, mode=""):
    report = sdfg.generate(str(folder), mode)
    text = re.sub(r"\s+", " ", open(report["source"]).read())
    return [c for c in re.findall(r"DOCC_ROCM_CHECK\((docc_rocm_(?:linear|layer_norm|\w*gemm\w*|reduce|elementwise\w*|cast|launch)\(.*?\))\);", text)]


class Block(torch.nn.Module):
    def forward(self, x, g, b, w1, b1, w2, b2):
        return x + F.linear(F.gelu(F.linear(F.layer_norm(x, (16,), g, b), w1, b1)), w2, b2)


def block_sdfg(dtype, rows):
    t = lambda *s: torch.randn(*s).to(dtype)
    return docc_torch.compile_torch(Block(), None, target="rocm").to_sdfg(t(rows, 16), t(16), t(16), t(64, 16), t(64), t(16, 64), t(16))


@pytest.mark.parametrize("rows", [5, 1])
@pytest.mark.parametrize("dtype,code", [(torch.float32, 2), (torch.bfloat16, 1)])
def test_a_feed_forward_block_is_three_calls(tmp_path, dtype, code, rows):
    s = block_sdfg(dtype, rows)
    s.schedule("rocm", options={"offload": "none"})
    assert [n["code"] for n in s.library_nodes()].count("GEMM") == 2      # the scheduled form keeps its nodes
    got = calls(s, tmp_path)
    rounds = (1, 2) if dtype == torch.bfloat16 else (0, 0)
    assert got == [f"docc_rocm_layer_norm(nullptr, {code}, {rows}, 16, (float) (1e-05), _x, _weight, _bias, _y)",
                   f"docc_rocm_linear(nullptr, {code}, 111, 112, {rows}, 64, 16, (float) __alpha, _a, 16, _b, 16, _bias, {code}, 16, nullptr, 2, {rounds[0]}, _y, {code})",
                   f"docc_rocm_linear(nullptr, {code}, 111, 112, {rows}, 16, 64, (float) __alpha, _a, 64, _b, 64, _bias, {code}, -1, _residual, {code}, {rounds[1]}, _y, {code})"]
    # every transient that is left is allocated before and freed behind its uses
    text = open(next(tmp_path.glob("*.cpp"))).read()
    assert text.count("docc_rocm_malloc_async(") == text.count("docc_rocm_free_async(") == 2


def test_instrumented_and_unfused_programs_keep_their_launches(tmp_path):
    s = block_sdfg(torch.float32, 5)
    s.schedule("rocm", options={"offload": "none"})
    assert "docc_rocm_linear" not in " ".join(calls(s, tmp_path / "ols", "ols"))
    s = block_sdfg(torch.float32, 5)
    s.schedule("rocm", options={"offload": "none", "fuse": False})
    assert "docc_rocm_linear" not in " ".join(calls(s, tmp_path / "apart"))


def two_layers(element, second_reader=False, factor="0.5"):
    b = StructuredSDFGBuilder("layers")
    for n in ("X", "W", "R", "Y", "Z"):
        b.add_container(n, element, True)
    for n in ("T0", "T1", "T2"):
        b.add_container(n, element, False, transient_bytes=32 * 16 * 8)
    b.add_gemm("X", "W", "T0", "1.0", "0.0", 32, 16, 8)
    b.add_elementwise_unary_op("sigmoid", "T0", "T1", [32, 16])
    b.add_elementwise_op("mul", "T0", "T1", "T2", [32, 16])
    b.add_elementwise_op("add", "T2", "R", "Y", [32, 16])
    if second_reader:
        b.add_elementwise_op("mul", "T0", factor, "Z", [32, 16])
    s = b.move()
    s.schedule("rocm", options={"offload": "none"})
    return s


def test_only_float_products_with_one_reader_are_merged(tmp_path):
    got = calls(two_layers(F32), tmp_path / "a")
    assert got == ["docc_rocm_linear(nullptr, 2, 111, 111, 32, 16, 8, (float) __alpha, _a, 8, _b, 16, nullptr, 2, 18, _residual, 2, 0, _y, 2)"]
    assert "docc_rocm_linear" not in " ".join(calls(two_layers(F64), tmp_path / "b"))
    assert "docc_rocm_linear" not in " ".join(calls(two_layers(F32, second_reader=True), tmp_path / "c"))


def bounded_product(bound):
    b = StructuredSDFGBuilder("bounded")
    for n in ("X", "W", "Y"):
        b.add_container(n, F32, True)
    b.add_container("T0", F32, False, transient_bytes=32 * 16 * 4)
    b.add_gemm("X", "W", "T0", "1.0", "0.0", 32, 16, 8)
    b.add_elementwise_op("maximum", "T0", bound, "Y", [32, 16])
    s = b.move()
    s.schedule("rocm", options={"offload": "none"})
    return s


# a bound is zero only where its text is the number: any other text goes into the code as it is written
@pytest.mark.parametrize("bound,relu", [("0.0", True), ("0", True), ("0.0f", True), ("-0.0", False), ("FLT_MAX", False), ("M_PI", False), ("(-1.5)", False),
                                        ("0.0 + 1.5", False), ("1.5", False)])
def test_the_larger_of_a_product_and_a_bound(tmp_path, bound, relu):
    got = " ".join(calls(bounded_product(bound), tmp_path))
    assert ("docc_rocm_linear" in got) == relu
    if not relu:
        assert bound in open(next(tmp_path.glob("*.cpp"))).read()


def test_factors_are_read_as_whole_numbers_only(tmp_path):
    b = StructuredSDFGBuilder("factors")
    for n in ("X", "W", "Y"):
        b.add_container(n, F32, True)
    for n in ("T0", "T1", "T2", "T3", "T4"):
        b.add_container(n, F32, False, transient_bytes=32 * 16 * 4)
    b.add_gemm("X", "W", "T0", "1.0", "0.0", 32, 16, 8)
    b.add_elementwise_op("mul", "T0", "0.7071067811865476 * 2", "T1", [32, 16])
    b.add_elementwise_unary_op("erf", "T1", "T2", [32, 16])
    b.add_elementwise_op("add", "T2", "1.0", "T3", [32, 16])
    b.add_elementwise_op("mul", "T0", "0.5", "T4", [32, 16])
    b.add_elementwise_op("mul", "T4", "T3", "Y", [32, 16])
    s = b.move()
    s.schedule("rocm", options={"offload": "none"})
    assert "docc_rocm_linear" not in " ".join(calls(s, tmp_path))


def test_an_empty_product_is_not_launched(tmp_path):
    # no columns: the leading dimension of W and Y is 0, which the launcher refuses; the GEMM node alone has always been guarded
    b = StructuredSDFGBuilder("empty")
    b.add_container("n", Scalar(PrimitiveType.Int64), True)
    for name in ("X", "W", "Y"):
        b.add_container(name, F32, True)
    b.add_container("T", F32, False, transient_bytes="32*n*4")
    b.add_gemm("X", "W", "T", "1.0", "0.0", 32, "n", 8)
    b.add_elementwise_unary_op("sigmoid", "T", "Y", [32, "n"])
    s = b.move()
    s.schedule("rocm", options={"offload": "none"})
    assert "docc_rocm_linear" in " ".join(calls(s, tmp_path))
    text = re.sub(r"\s+", " ", open(next(tmp_path.glob("*.cpp"))).read())
    assert "if ((32) != 0 && (n) != 0) DOCC_ROCM_CHECK(docc_rocm_linear(" in text


@pytest.mark.parametrize("between", [False, True])
def test_an_operand_that_a_download_frees_stays_with_its_product(tmp_path, between):
    # H is computed, multiplied and copied back; the copy releases its device buffer. Where that happens between the product and the
    # elementwise node behind it, the product must not move down to that node
    b = StructuredSDFGBuilder("download")
    for n in ("X", "W", "H", "Y"):
        b.add_container(n, F32, True)
    for n in ("T0", "T1"):
        b.add_container(n, F32, False, transient_bytes=32 * 16 * 4)
    b.add_elementwise_unary_op("relu", "X", "H", [32, 8])
    b.add_gemm("H", "W", "T0", "1.0", "0.0", 32, 16, 8)
    b.add_elementwise_unary_op("sigmoid", "T0", "T1", [32, 16])
    b.add_elementwise_op("mul", "T0", "T1", "Y", [32, 16])
    s = b.move()
    s.schedule("rocm")
    form = json.loads(s.to_json())
    blocks = form["root"]["children"]
    node = lambda e: e["dataflow"]["library_node"]
    reads = lambda e, name: any(i.get("data", "").endswith(name) for i in e["dataflow"]["inputs"])
    copy = next(e for e in blocks if node(e).get("transfer_direction") == -1 and reads(e, "_H"))
    free = next(e for e in blocks if node(e).get("transfer_direction") == 0 and node(e).get("buffer_lifecycle") == -1 and reads(e, "_H"))
    if between:
        node(copy)["buffer_lifecycle"] = -1
        blocks.remove(copy)
        blocks[blocks.index(free)] = copy
    names = [node(e)["code"] for e in blocks]
    assert blocks.index(copy) > names.index("GEMM") if between else blocks.index(copy) < names.index("GEMM")
    got = calls(StructuredSDFG.parse(json.dumps(form)), tmp_path)
    assert ("docc_rocm_linear" in " ".join(got)) == (not between)


@pytest.mark.parametrize("beta,read", [("0.0", False), ("0", False), ("0.0f", False), ("0.5", True), ("M_PI", True), ("0.0 + 1.0", True)])
def test_c_is_read_unless_beta_is_the_number_zero(tmp_path, beta, read):
    b = StructuredSDFGBuilder("beta")
    for n in ("X", "W", "C", "Y"):
        b.add_container(n, F32, True)
    b.add_gemm("X", "W", "C", "1.0", beta, 32, 16, 8)
    b.add_elementwise_unary_op("sigmoid", "C", "Y", [32, 16])
    s = b.move()
    s.schedule("rocm")
    assert s.loop_report()["H2D"] == (3 if read else 2)


class ConvBlock(torch.nn.Module):
    def __init__(self, tail):
        super().__init__()
        self.tail = tail

    def forward(self, x, r, w, b):
        return self.tail(F.conv2d(x, w, b, padding=1), r)


CONV = "2, 8, 6, 6, 16, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, (int64_t) (1), X, W, B"


@pytest.mark.parametrize("tail,emitted", [
    (lambda y, r: torch.relu(y), f"{CONV}, nullptr, 2, _y"),
    (lambda y, r: torch.relu(y + r), f"{CONV}, _residual, 2, _y"),
    (lambda y, r: torch.relu(r + y), f"{CONV}, _residual, 2, _y"),
    (lambda y, r: y + r, f"{CONV}, _residual, -1, _y"),
    (lambda y, r: torch.sigmoid(y), None),                     # no activation of the store
    (lambda y, r: torch.relu(y) + y, None),                    # a second reader
    (lambda y, r: torch.relu(y - r), None),
    (lambda y, r: torch.relu(y + y), None),
    (lambda y, r: torch.relu(y + r), "repeated"),
])
def test_a_convolution_with_the_block_behind_it(tmp_path, tail, emitted):
    images = 1 if emitted == "repeated" else 2          # a residual of one image for both
    emitted = emitted if images == 2 else None
    s = docc_torch.compile_torch(ConvBlock(tail), None, target="rocm").to_sdfg(torch.randn(2, 8, 6, 6), torch.randn(images, 16, 6, 6), torch.randn(16, 8, 3, 3), torch.randn(16))
    s.schedule("rocm", options={"offload": "none"})
    assert [n["code"] for n in s.library_nodes()].count("ml::Conv") == 1      # the scheduled form keeps its nodes
    text = re.sub(r"\s+", " ", open(s.generate(str(tmp_path))["source"]).read())
    if emitted:
        assert f"docc_rocm_conv2d_f32_chain(nullptr, {emitted}, __ws, __ws_bytes)" in text and "elementwise" not in text and text.count("docc_rocm_malloc_async(") == 1
    else:
        assert "docc_rocm_conv2d_f32_chain" not in text and "docc_rocm_conv2d_f32_pads(" in text


@pytest.mark.parametrize("shape,merged", [(["n", "256"], "docc_rocm_softmax_f32_host(nullptr, n, 256, _x, _y)"), (["65536", "256"], "docc_rocm_softmax_f32_host(nullptr, 65536, 256, _x, _y)"),
                                          (["64", "256"], None)])
@pytest.mark.parametrize("reader", [False, True])
def test_a_softmax_between_an_upload_and_a_download(tmp_path, shape, merged, reader):
    """Large host arrays go through docc_rocm_softmax_host; not those that are known to be small, nor results that another node reads on the device."""
    b = StructuredSDFGBuilder("rows")
    b.add_container("n", Scalar(PrimitiveType.Int64), True)
    for name in ("X", "Y", "Z"):
        b.add_container(name, F32, True)
    b.add_reduce_op("softmax", "X", "Y", shape, [1])
    if reader:
        b.add_elementwise_unary_op("relu", "Y", "Z", shape)
    s = b.move()
    s.schedule("rocm", options={"fuse_maps": False})
    text = re.sub(r"\s+", " ", open(s.generate(str(tmp_path))["source"]).read())
    if merged and not reader:
        assert merged in text and "memcpy" not in text and "malloc" not in text
    else:
        assert "_host(" not in text and "docc_rocm_softmax_f32(nullptr, " in text and text.count("docc_rocm_memcpy_h2d_async(") == 1


@pytest.mark.parametrize("rows,width,merged", [(8, 64, True), (1, 64, True), (16, 64, True), (17, 64, False), (8, 16, False)])
def test_a_layer_norm_and_the_layer_behind_it(tmp_path, rows, width, merged):
    class Layer(torch.nn.Module):
        def forward(self, x, g, b, w, c):
            return F.relu(F.linear(F.layer_norm(x, (width,), g, b), w, c))

    t = lambda *s: torch.randn(*s).bfloat16()
    s = docc_torch.compile_torch(Layer(), None, target="rocm").to_sdfg(t(rows, width), t(width), t(width), t(48, width), t(48))
    s.schedule("rocm", options={"offload": "none"})
    text = re.sub(r"\s+", " ", open(s.generate(str(tmp_path))["source"]).read())
    if merged:
        assert f"docc_rocm_norm_linear(nullptr, 1, {rows}, 48, {width}, (float) (1e-05), _x, _weight, _norm_bias, (float) __alpha, _b, {width}, _bias, 1, 2, nullptr, 2, 1, _scratch, _y, 1)" in text
        assert "docc_rocm_layer_norm" not in text and "docc_rocm_linear" not in text
        assert text.count("docc_rocm_malloc_async(") == text.count("docc_rocm_free_async(") == 1
    else:
        assert "docc_rocm_norm_linear" not in text and "docc_rocm_layer_norm(" in text and "docc_rocm_linear(" in text


# the one launch of both leaves the normalised rows nowhere: a layer that has them as its residual or as its weights too keeps them
@pytest.mark.parametrize("again", ["residual", "weights"])
def test_a_layer_norm_that_its_layer_reads_twice(tmp_path, again):
    class Layer(torch.nn.Module):
        def forward(self, x, g, b, w, c):
            h = F.layer_norm(x, (64,), g, b)
            if again == "residual":
                return h + F.linear(h, w, c)
            return F.relu(F.linear(h, h, c))

    t = torch.randn
    s = docc_torch.compile_torch(Layer(), None, target="rocm").to_sdfg(t(8, 64), t(64), t(64), t(64, 64), t(64 if again == "residual" else 8))
    s.schedule("rocm", options={"offload": "none"})
    text = re.sub(r"\s+", " ", open(s.generate(str(tmp_path))["source"]).read())
    assert "docc_rocm_norm_linear" not in text and "docc_rocm_layer_norm(" in text
