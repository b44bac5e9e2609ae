"""docc_rocm_linear (a product with bias, activation, roundings and residual behind it) and docc_rocm_layer_norm, and the programs
the code generator emits them for. Against float64 on the CPU, with the roundings to bf16 that the chain asks for."""
import ctypes

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from docc_amd import runtime as rt

pytestmark = pytest.mark.gpu

ACTS = {None: -1, "abs": 0, "relu": 2, "sigmoid": 3, "tanh": 5, "gelu": 16, "gelu_tanh": 17, "silu": 18}
REF = {None: lambda x: x, "abs": torch.abs, "relu": torch.relu, "sigmoid": torch.sigmoid, "tanh": torch.tanh, "gelu": F.gelu,
       "gelu_tanh": lambda x: F.gelu(x, approximate="tanh"), "silu": F.silu}
TYPE = {torch.bfloat16: 1, torch.float32: 2}


def ptr(t):
    return ctypes.c_void_p(t.data_ptr() if t is not None else None)


def linear(a, w, trans_b, bias, act, residual, rounding, out_dtype, y=None):
    m, k = a.shape
    n = w.shape[0] if trans_b else w.shape[1]
    y = y if y is not None else torch.full((m, n), float("nan"), device="cuda", dtype=out_dtype)
    rt.call("docc_rocm_linear", 0, TYPE[a.dtype], rt.NO_TRANS, rt.TRANS if trans_b else rt.NO_TRANS, m, n, k, 1.0, ptr(a), k, ptr(w), w.shape[1],
            ptr(bias), TYPE[bias.dtype] if bias is not None else 2, ACTS[act], ptr(residual), TYPE[residual.dtype] if residual is not None else 2,
            rounding, ptr(y), TYPE[out_dtype])
    torch.cuda.synchronize()
    return y


def reference(a, w, trans_b, bias, act, residual, rounding):
    v = a.double().cpu() @ (w.double().cpu().T.contiguous() if trans_b else w.double().cpu())
    if bias is not None:
        v = v + bias.double().cpu()
    if rounding & 1:
        v = v.float().bfloat16().double()
    v = REF[act](v)
    if residual is not None:
        if rounding & 2:
            v = v.float().bfloat16().double()
        v = v + residual.double().cpu()
    return v


# rows: matrix-vector, few-row kernels, tiles of 64 / 128 / 256 with ragged edges, K in parts; columns off a vector of eight too
@pytest.mark.parametrize("waves", ["", "0"])       # 0: without the kernels that cut K between wavefronts, which take most of the few rows
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(1, 512, 512), (2, 1024, 2048), (8, 4096, 2048), (17, 8192, 1024), (64, 256, 1024), (100, 72, 96), (129, 200, 64),
                                   (130, 77, 33), (384, 1032, 512), (1000, 136, 4096), (2050, 1160, 128), (4100, 4104, 128)])
def test_linear_over_the_launchers_forms(monkeypatch, dtype, m, n, k, waves):
    if waves:
        monkeypatch.setenv("DOCC_ROCM_GEMM_WAVES", waves)
    gen = torch.Generator().manual_seed(m * 31 + n)
    a = torch.randn(m, k, generator=gen).to(dtype).cuda()
    w = (torch.randn(n, k, generator=gen) * k ** -0.5).to(dtype).cuda()
    bias = torch.randn(n, generator=gen).to(dtype).cuda()
    res = torch.randn(m, n, generator=gen).to(dtype).cuda()
    for act, b, r, rounding in (("gelu", bias, None, 1), (None, bias, res, 2), ("relu", None, res, 3)):
        rounding = rounding if dtype == torch.bfloat16 else 0
        ref = reference(a, w, True, b, act, r, rounding)
        got = linear(a, w, True, b, act, r, rounding, dtype)
        # the fp32 sums: k products of size 1 / sqrt(k), each rounded at 2^-24, the error growing with sqrt(k): 2^-24 * sqrt(4096) * a few
        # at most, whatever the size of the result. bf16 on top of that: a last
        # bit (at most 2^-7 of the value) of the result, and one of the value that is rounded in between where the fp32 sum and the exact
        # one lie on different sides of a boundary - before the activation, whose slope is at most 1.13, or behind it, where it is smaller
        err = (got.double().cpu() - ref).abs()
        between = reference(a, w, True, b, None, None, 0).abs()
        bound = 2e-5 * (1 + ref.abs()) + (0 if dtype == torch.float32 else 2.0 ** -7 * (1.13 * between + ref.abs()))
        assert bool((err <= bound).all()), (act, float((err / bound).max()))


# K cut between the wavefronts of a work-group (csrc/kernels/gemm_waves.hip), in pieces of 64 or 128 bytes of a row that four or eight wavefronts take in turn: less
# than a piece, a part of one behind many, more pieces than are on their way at once, ragged tiles - and rows of A and B that are longer than K
@pytest.mark.parametrize("tile", ["16", "32", "64", "1"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k,ld", [(1, 8, 8, 8), (2, 24, 64, 64), (7, 40, 72, 80), (8, 16, 1032, 1032), (9, 520, 200, 208), (16, 72, 4168, 4168), (17, 8, 136, 136),
                                      (32, 264, 2056, 2064), (65, 136, 520, 520), (130, 72, 264, 272)])
def test_linear_cut_between_wavefronts(monkeypatch, tile, dtype, m, n, k, ld):
    monkeypatch.setenv("DOCC_ROCM_GEMM_WAVES", tile)
    gen = torch.Generator().manual_seed(m * 31 + n)
    a, w = torch.randn(m, ld, generator=gen).to(dtype).cuda(), (torch.randn(n, ld, generator=gen) * k ** -0.5).to(dtype).cuda()
    a[:, k:], w[:, k:] = float("nan"), float("inf")           # behind the rows: not read, or dropped
    bias, res = torch.randn(n, generator=gen).to(dtype).cuda(), torch.randn(m, n, generator=gen).to(dtype).cuda()
    for act, b, r in (("gelu", bias, None), (None, None, res), ("relu", bias, res)):
        y = torch.full((m, n), float("nan"), device="cuda", dtype=dtype)
        rt.call("docc_rocm_linear", 0, TYPE[dtype], rt.NO_TRANS, rt.TRANS, m, n, k, 0.5, ptr(a), ld, ptr(w), ld, ptr(b), TYPE[dtype], ACTS[act], ptr(r), TYPE[dtype], 0,
                ptr(y), TYPE[dtype])
        torch.cuda.synchronize()
        ref = reference(a[:, :k] * 0.5, w[:, :k], True, b, act, r, 0)
        bound = 2e-5 * (1 + ref.abs()) + (0 if dtype == torch.float32 else 2.0 ** -7 * ref.abs())      # as above, nothing rounded in between
        err = (y.double().cpu() - ref).abs()
        assert bool((err <= bound).all()), (act, float((err / bound).max()))


# the layer norm in front of it in the same launch: a piece and a part of one, 4 and 8 vectors a lane and one short of that, and shapes that keep their two launches
@pytest.mark.parametrize("tile", ["16", "32"])      # 32: two launches
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(1, 8, 64), (7, 40, 72), (8, 4096, 2048), (5, 24, 1016), (9, 72, 1024), (16, 520, 256), (16, 8, 2048), (8, 16, 4096), (3, 16, 4104), (17, 16, 128),
                                   (4, 8, 16)])
def test_layer_norm_and_linear_as_one(monkeypatch, tile, dtype, m, n, k):
    monkeypatch.setenv("DOCC_ROCM_GEMM_WAVES", tile)
    gen = torch.Generator().manual_seed(m * 31 + n)
    x = (torch.randn(m, k, generator=gen) * 3 + 5).to(dtype).cuda()
    gain, shift = (1 + torch.randn(k, generator=gen) * 0.1).to(dtype).cuda(), torch.randn(k, generator=gen).to(dtype).cuda()
    w, bias = (torch.randn(n, k, generator=gen) * k ** -0.5).to(dtype).cuda(), torch.randn(n, generator=gen).to(dtype).cuda()
    res = torch.randn(m, n, generator=gen).to(dtype).cuda()
    for g, b, act, r in ((gain, shift, "gelu", None), (None, None, None, res), (gain, None, "relu", res)):
        y, scratch = torch.full((m, n), float("nan"), device="cuda", dtype=dtype), torch.empty_like(x)
        rt.call("docc_rocm_norm_linear", 0, TYPE[dtype], m, n, k, 1e-5, ptr(x), ptr(g), ptr(b), 1.0, ptr(w), k, ptr(bias), TYPE[dtype], ACTS[act], ptr(r), TYPE[dtype], 0,
                ptr(scratch), ptr(y), TYPE[dtype])
        torch.cuda.synchronize()
        h = F.layer_norm(x.double().cpu(), (k,), g.double().cpu() if g is not None else None, b.double().cpu() if b is not None else None, 1e-5).to(dtype)
        ref = reference(h, w, True, bias, act, r, 0)
        # as above; the normalised rows of both sides may lie on different sides of a rounding to bf16 here and there: k terms of 2^-8 k^-1/2 at most a few times that
        bound = 2e-5 * (1 + ref.abs()) + (0 if dtype == torch.float32 else 2.0 ** -7 * (1 + ref.abs()))
        err = (y.double().cpu() - ref).abs()
        assert bool((err <= bound).all()), (act, float((err / bound).max()))


# the rows in place, and the normalised rows as residual or as weights: what two launches give
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,k", [(1, 64), (8, 2048), (16, 1024)])
def test_layer_norm_and_linear_on_operands_that_overlap(dtype, m, k):
    gen = torch.Generator().manual_seed(k)
    x = (torch.randn(m, k, generator=gen) * 3 + 5).to(dtype).cuda()
    w, bias = (torch.randn(k, k, generator=gen) * k ** -0.5).to(dtype).cuda(), torch.randn(k, generator=gen).to(dtype).cuda()
    h = F.layer_norm(x.double().cpu(), (k,), None, None, 1e-5).to(dtype)
    for case in ("in place", "normed residual", "normed weights"):
        n = m if case == "normed weights" else k
        scratch, y = torch.full_like(x, float("nan")), x.clone() if case == "in place" else torch.full((m, n), float("nan"), device="cuda", dtype=dtype)
        X, W, r = (y, w, y) if case == "in place" else (x, w, scratch) if case == "normed residual" else (x, scratch, None)
        rt.call("docc_rocm_norm_linear", 0, TYPE[dtype], m, n, k, 1e-5, ptr(X), None, None, 1.0, ptr(W), k, ptr(bias[:n]), TYPE[dtype], -1, ptr(r), TYPE[dtype], 0,
                ptr(scratch), ptr(y), TYPE[dtype])
        torch.cuda.synchronize()
        ref = reference(h, h if case == "normed weights" else w, True, bias[:n], None, {"in place": x, "normed residual": h, "normed weights": None}[case], 0)
        bound = 2e-5 * (1 + ref.abs()) + (0 if dtype == torch.float32 else 2.0 ** -7 * (1 + ref.abs()))      # as above
        if case == "normed weights":      # k products of size 1, and their differences by the rows' roundings to bf16
            bound = bound + (4e-6 if dtype == torch.float32 else 2.0 ** -7) * k ** 0.5 * 4
        err = (y.double().cpu() - ref).abs()
        assert bool((err <= bound).all()), (case, float((err / bound).max()))


# every tile with the chain in its store, ragged at both edges and along K where the tile allows it
@pytest.mark.parametrize("cfg,dtype,k", [("128x128x32x4x4", torch.bfloat16, 104), ("128x128x64x4x4", torch.bfloat16, 328), ("128x256x64x4x3", torch.bfloat16, 328),
                                         ("256x256x32x4x4q", torch.bfloat16, 192), ("64x64x16x4x4", torch.float32, 84), ("128x128x32x4x3", torch.float32, 84),
                                         ("128x256x32x4x2", torch.float32, 84), ("256x256x32x4x2", torch.float32, 84)])
@pytest.mark.parametrize("trans_b", [True, False])
def test_linear_tiles(monkeypatch, cfg, dtype, k, trans_b):
    monkeypatch.setenv("DOCC_ROCM_GEMM_CFG", cfg)
    gen = torch.Generator().manual_seed(k)
    for m, n in ((256, 256), (259, 520), (65, 264)):
        a = torch.randn(m, k, generator=gen).to(dtype).cuda()
        w = (torch.randn(*((n, k) if trans_b else (k, n)), generator=gen) * k ** -0.5).to(dtype).cuda()
        bias, res = torch.randn(n, generator=gen).to(dtype).cuda(), torch.randn(m, n, generator=gen).to(dtype).cuda()
        got = linear(a, w, trans_b, bias, "silu", res, 0, torch.float32).double().cpu()
        assert float((got - reference(a, w, trans_b, bias, "silu", res, 0)).abs().max()) <= 2e-5     # fp32 throughout: sums of at most 328 terms


@pytest.mark.parametrize("act", list(ACTS))
@pytest.mark.parametrize("trans_b", [True, False])
def test_linear_activations(act, trans_b):
    gen = torch.Generator().manual_seed(5)
    a = torch.randn(192, 64, generator=gen).cuda()
    w = (torch.randn(136, 64, generator=gen) * 0.4).cuda()
    w = w if trans_b else w.T.contiguous()
    bias = torch.randn(136, generator=gen).cuda()
    got = linear(a, w, trans_b, bias, act, None, 0, torch.float32).double().cpu()
    ref = reference(a, w, trans_b, bias, act, None, 0)
    # |x| up to about 15; sums of 64 terms in fp32 (2e-6) through slopes of at most 1.13
    assert float((got - ref).abs().max()) <= 1e-5


# the chain in the store, behind parts of K, behind a matrix-vector product, and element by element (n = 77: no whole vectors)
CHAINS = [(256, 256, "0"), (256, 256, "4"), (1, 4096, "0"), (130, 77, "0")]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,splits", CHAINS)
def test_roundings_in_between(monkeypatch, dtype, m, n, splits):
    """Whole numbers: every fp32 sum is exact, most of them have more bits than a bf16 value, and each rounding shows."""
    monkeypatch.setenv("DOCC_ROCM_GEMM_SPLITK", splits)
    gen = torch.Generator().manual_seed(m + n)
    draw = lambda *shape: torch.randint(-7, 8, shape, generator=gen).float()
    a, w, bias, res = draw(m, 512), draw(n, 512), draw(n), draw(m, n)
    at = lambda t: t.to(dtype).cuda()
    seen = []
    for act in (None, "relu", "abs"):
        for rounding in (0, 1, 2, 3):
            want = reference(a, w, True, bias, act, res, rounding).float()
            got = linear(at(a), at(w), True, at(bias), act, at(res), rounding, torch.float32).cpu()
            assert torch.equal(got, want), (act, rounding)
            seen.append(want)
            # Y may be the residual itself
            y = res.cuda()
            assert torch.equal(linear(at(a), at(w), True, at(bias), act, y, rounding, torch.float32, y).cpu(), want)
        assert not torch.equal(seen[-4], seen[-3]) and not torch.equal(seen[-4], seen[-2])


@pytest.mark.parametrize("n,splits", [(256, "0"), (77, "0")])
def test_activations_of_values_that_are_not_finite(monkeypatch, n, splits):
    monkeypatch.setenv("DOCC_ROCM_GEMM_SPLITK", splits)
    inf = float("inf")
    x = torch.tensor([inf, -inf, float("nan"), 1e30, -1e30, 3e38, -3e38, 100.0, -100.0, 12.0, -12.0, 0.0])
    a, w = torch.zeros(len(x), 64), torch.zeros(n, 64)
    a[:, 0], w[:, 0] = x, 1
    # as the nodes spell them, in fp32: -inf times a factor that is 0 is a NaN
    spelled = {None: x, "abs": x.abs(), "relu": torch.fmax(x, torch.zeros(())), "sigmoid": 1 / (1 + torch.exp(-x)), "tanh": torch.tanh(x),
               "gelu": 0.5 * x * (1 + torch.erf(x * 0.7071067811865476)), "gelu_tanh": 0.5 * x * (1 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x * x * x))),
               "silu": x * (1 / (1 + torch.exp(-x)))}
    for act, want in spelled.items():
        got = linear(a.cuda(), w.cuda(), True, None, act, None, 0, torch.float32).cpu()
        # (1e-5: the gelu of -12 and -100, zero where it cancels and 1e-32 where it does not)
        assert torch.allclose(got, want[:, None].expand(-1, n), rtol=1e-6, atol=1e-5, equal_nan=True), (act, got[:, 0], want)


def test_a_captured_layer_norm_in_slices_replays():
    # its sums are in the stream's buffer, which the program's own calls on that stream use between the replays
    gen = torch.Generator().manual_seed(1)
    x, other = (torch.randn(3, 40000, generator=gen).cuda() for _ in range(2))
    y, z, want = torch.empty_like(x), torch.empty_like(x), torch.empty_like(x)
    norm = lambda x, y, s: rt.call("docc_rocm_layer_norm", s, 2, 3, 40000, 1e-5, ptr(x), None, None, ptr(y))
    norm(x, want, 0)
    torch.cuda.synchronize()
    s = rt.stream_create()
    try:
        norm(other, z, s)
        with rt.Graph.capture(s) as graph:
            norm(x, y, s)
        for _ in range(3):
            y.fill_(float("nan"))
            torch.cuda.synchronize()
            graph.launch()
            norm(other, z, s)
            rt.stream_sync(s)
            assert torch.equal(y, want)
        graph.destroy()
    finally:
        rt.stream_destroy(s)


@pytest.mark.parametrize("rows,cols", [(700, 4), (1100, 256), (3, 250), (5, 1024), (3, 4097), (2, 20000)])
def test_layer_norm_of_values_far_from_one(rows, cols):
    # roots from 0 to infinity, some where the quotient is not formed from the reciprocal; whole numbers times a power of two keep the sums exact
    gen = torch.Generator().manual_seed(cols)
    half = torch.randint(1, 8, (rows, cols // 2), generator=gen).float().numpy()
    x = np.concatenate([half, -half, np.zeros((rows, cols % 2), np.float32)], 1)
    for scale in (2.0 ** -120, 2.0 ** -66, 2.0 ** -40, 2.0 ** 40, 2.0 ** 62, 2.0 ** 100):
        d = x * np.float32(scale)
        dx = torch.from_numpy(d).cuda()
        y = torch.full_like(dx, 5.0)
        rt.call("docc_rocm_layer_norm", 0, 2, rows, cols, 0.0, ptr(dx), None, None, ptr(y))
        torch.cuda.synchronize()
        with np.errstate(all="ignore"):
            want = d / np.sqrt(np.square(d).sum(1, keepdims=True) / np.float32(cols))
        assert np.array_equal(y.cpu().numpy(), want, equal_nan=True), scale


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,cols", [(700, 3), (600, 8), (70, 64), (1100, 256), (6, 250), (6, 2048), (6, 9001), (6, 16384), (6, 20000), (6, 33333)])
def test_layer_norm_in_place_and_with_values_that_are_not_finite(dtype, rows, cols):
    gen = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, cols, generator=gen).to(dtype).cuda()
    w, b = torch.randn(cols, generator=gen).to(dtype).cuda(), torch.randn(cols, generator=gen).to(dtype).cuda()

    def norm(x, y):
        rt.call("docc_rocm_layer_norm", 0, TYPE[dtype], rows, cols, 1e-5, ptr(x), ptr(w), ptr(b), ptr(y))
        torch.cuda.synchronize()
        return y

    plain = norm(x, torch.empty_like(x))
    same = x.clone()
    assert torch.equal(norm(same, same), plain)
    x[1, cols // 2], x[3, 0], x[4, cols - 1] = float("inf"), float("nan"), -float("inf")
    got = norm(x, torch.empty_like(x))
    spoilt = torch.zeros(rows, dtype=torch.bool, device="cuda")
    spoilt[[1, 3, 4]] = True
    assert bool(got[spoilt].isnan().all()) and torch.equal(got[~spoilt], plain[~spoilt])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,cols", [(1, 1), (700, 1), (1, 2), (513, 3), (1000, 4), (300, 5), (259, 8), (130, 16), (65, 17), (40, 32), (30, 40), (17, 64), (9, 100), (9, 128),
                                       (9, 129), (5, 248), (5, 256), (1, 8), (3, 250), (5, 1000), (1025, 256), (2000, 1024), (8, 2048), (1030, 2048), (7, 4096), (5, 4097), (3, 8192),
                                       (2, 16384), (2, 9001)])
def test_layer_norm_over_row_lengths(dtype, rows, cols):
    gen = torch.Generator().manual_seed(cols)
    x = (torch.randn(rows, cols, generator=gen) * 3 + 1).to(dtype).cuda()
    w, b = torch.randn(cols, generator=gen).to(dtype).cuda(), torch.randn(cols, generator=gen).to(dtype).cuda()
    for weight, bias in ((w, b), (None, None), (w, None)):
        y = torch.full_like(x, float("nan"))
        rt.call("docc_rocm_layer_norm", 0, TYPE[dtype], rows, cols, 1e-5, ptr(x), ptr(weight), ptr(bias), ptr(y))
        torch.cuda.synchronize()
        up = lambda t: None if t is None else t.double().cpu()
        ref = F.layer_norm(up(x), (cols,), up(weight), up(bias), 1e-5)
        err = (y.double().cpu() - ref).abs()
        bound = 1e-5 * (1 + ref.abs()) if dtype == torch.float32 else 2.0 ** -8 * (1e-3 + ref.abs())
        assert bool((err <= bound).all()), float((err / bound).max())


# rows in slices: one and several of them, the last one short, more rows than would get more than one each; as many slices as there can be
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,cols", [(1, 9000), (2, 9001), (700, 8200), (1, 300000), (3, 65537), (300, 16400)])
def test_layer_norm_of_long_rows_in_slices(monkeypatch, dtype, rows, cols):
    monkeypatch.setenv("DOCC_ROCM_LAYERNORM", "slices")
    test_layer_norm_over_row_lengths(dtype, rows, cols)


@pytest.mark.parametrize("rows,cols", [(700, 3), (700, 4), (300, 8), (200, 24), (90, 50), (60, 128), (1100, 256), (3, 250), (5, 1024), (2, 4096), (3, 4097), (2, 16384), (2, 20000), (3, 33333)])
def test_layer_norm_divides_by_the_root(rows, cols):
    # small whole numbers whose mean is one too: both sums are exact in fp32 whatever their order, what is left is a division by cols, the
    # root and one division an element, each rounded once
    gen = torch.Generator().manual_seed(cols)
    half = torch.randint(-7, 8, (rows, cols // 2), generator=gen).float()
    x = 3 + torch.cat([half, -half, torch.zeros(rows, cols % 2)], 1)[:, torch.randperm(cols, generator=gen)]
    d = x.numpy() - 3       # (numpy rounds each operation once; torch divides a tensor by a number through its reciprocal)
    want = d / np.sqrt(np.square(d).sum(1, keepdims=True) / np.float32(cols) + np.float32(1e-5))
    dx = x.cuda()
    y = torch.full_like(dx, float("nan"))
    rt.call("docc_rocm_layer_norm", 0, 2, rows, cols, 1e-5, ptr(dx), None, None, ptr(y))
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy(), want)


class Block(torch.nn.Module):
    def __init__(self, width, approximate):
        super().__init__()
        self.width, self.approximate = width, approximate

    def forward(self, x, g, b, w1, b1, w2, b2):
        h = F.layer_norm(x, (self.width,), g, b)
        return x + F.linear(F.gelu(F.linear(h, w1, b1), approximate=self.approximate), w2, b2)


@pytest.mark.parametrize("dtype,tokens,width,approximate", [(torch.float32, 96, 64, "none"), (torch.bfloat16, 200, 128, "tanh"), (torch.bfloat16, 1, 64, "none"),
                                                            (torch.bfloat16, 8, 2048, "none"), (torch.float32, 5, 100, "tanh")])
def test_block_program(dtype, tokens, width, approximate):
    import docc_amd.torch as docc_torch

    gen = torch.Generator().manual_seed(width)
    rand = lambda *s, scale=1.0: (torch.randn(*s, generator=gen) * scale).to(dtype).cuda()
    args = (rand(tokens, width), rand(width), rand(width), rand(4 * width, width, scale=width ** -0.5), rand(4 * width), rand(width, 4 * width, scale=0.5 * width ** -0.5), rand(width))
    got = docc_torch.compile_torch(Block(width, approximate), None, target="rocm")(*args)
    ref = Block(width, approximate)(*[t.double().cpu() for t in args])
    assert got.dtype == dtype and got.shape == ref.shape
    err = float((got.double().cpu() - ref).norm() / ref.norm())
    assert err <= (1e-5 if dtype == torch.float32 else 1e-2), err     # bf16: the three intermediate tensors are rounded to bf16


class NormedResidual(torch.nn.Module):
    def forward(self, x, g, b, w, c):
        h = F.layer_norm(x, (256,), g, b)
        return h + F.linear(h, w, c)


# the residual behind a layer is the layer norm in front of it
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens", [1, 8, 17])
def test_program_with_the_normalised_rows_as_residual(dtype, tokens):
    import docc_amd.torch as docc_torch

    gen = torch.Generator().manual_seed(tokens)
    rand = lambda *s: torch.randn(*s, generator=gen).to(dtype).cuda()
    args = (rand(tokens, 256), rand(256), rand(256), rand(256, 256) / 16, rand(256))
    got = docc_torch.compile_torch(NormedResidual(), None, target="rocm")(*args)
    ref = NormedResidual()(*[t.double().cpu() for t in args])
    err = float((got.double().cpu() - ref).norm() / ref.norm())
    assert err <= (1e-5 if dtype == torch.float32 else 1e-2), err     # as above, with two tensors in between
