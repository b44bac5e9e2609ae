"""Products whose operands are off the vectors of the asynchronous kernels (packed first, csrc/kernels/gemm_pack.hip) and products whose
K is cut into parts of different lengths. Against float64 on the CPU."""
import pytest
import torch

from docc_amd import runtime as rt

pytestmark = pytest.mark.gpu

KINDS = {"f64": (torch.float64, rt.dgemm, 2.0 ** -52), "f32": (torch.float32, rt.sgemm, 2.0 ** -23), "bf16": (torch.bfloat16, rt.bf16gemm_f32, 2.0 ** -23)}


def check(kind, m, n, k, ta, tb, alpha=1.0, beta=0.0, pad=0):
    dtype, gemm, eps = KINDS[kind]
    out = torch.float32 if kind == "bf16" else dtype
    gen = torch.Generator().manual_seed(m * 7 + n * 3 + k)
    # integers of a few bits: every sum is exact in fp32, so the result must be too whatever the order (k * 9 < 2^24)
    draw = lambda r, c: torch.randint(-3, 4, (r, c), generator=gen).to(dtype)
    a, b = draw(k, m) if ta else draw(m, k), draw(n, k) if tb else draw(k, n)
    # (leading dimensions larger than the rows, NaN between: nothing outside the operands takes part)
    wide = lambda t: torch.cat([t, torch.full((t.shape[0], pad), float("nan"), dtype=dtype)], 1).contiguous().cuda()
    da, db = wide(a), wide(b)
    c = torch.randint(-3, 4, (m, n), generator=gen).to(out).cuda()
    ref = alpha * ((a.double().T if ta else a.double()) @ (b.double().T if tb else b.double())) + (beta * c.double().cpu() if beta else 0)
    gemm(m, n, k, alpha, da.data_ptr(), da.shape[1], db.data_ptr(), db.shape[1], beta, c.data_ptr(), n,
         trans_a=rt.TRANS if ta else rt.NO_TRANS, trans_b=rt.TRANS if tb else rt.NO_TRANS)
    torch.cuda.synchronize()
    assert torch.equal(c.double().cpu(), ref), float((c.double().cpu() - ref).abs().max())


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("m,n,k,pad", [(65, 63, 65, 0), (1, 129, 64, 1), (130, 40, 1, 0), (67, 131, 127, 3), (96, 80, 72, 1), (200, 17, 193, 0), (33, 300, 1025, 0)])
def test_operands_off_the_vectors(monkeypatch, kind, ta, tb, m, n, k, pad):
    monkeypatch.setenv("DOCC_ROCM_GEMM_PACK", "1")
    check(kind, m, n, k, ta, tb, pad=pad)


@pytest.mark.parametrize("kind", list(KINDS))
def test_packed_products_by_size_alone(kind):
    for m, n, k, tb in ((517, 403, 301, False), (40, 50, 3001, True), (700, 301, 255, True)):
        check(kind, m, n, k, False, tb, alpha=2.0, beta=-1.0)


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("m,n,k", [(100, 104, 1000), (64, 128, 4264), (152, 200, 8016), (40, 320, 2056), (16, 16, 704)])
def test_parts_of_different_lengths(monkeypatch, kind, m, n, k):
    for waves in (None, "0"):       # 0: not between the wavefronts of a work-group, which most of these are chosen for
        if waves:
            monkeypatch.setenv("DOCC_ROCM_GEMM_WAVES", waves)
        for tb in (False, True):
            check(kind, m, n, k, False, tb)
        check(kind, m, n, k, True, False, alpha=0.5, beta=1.0)


@pytest.mark.parametrize("kind", list(KINDS))
def test_a_packed_product_in_a_capture_replays(monkeypatch, kind):
    """The packed operands' block belongs to the graph: replays between products of the program's own, which take blocks of that size too."""
    monkeypatch.setenv("DOCC_ROCM_GEMM_PACK", "1")
    dtype, gemm, _ = KINDS[kind]
    out = torch.float32 if kind == "bf16" else dtype
    m, n, k = 130, 67, 333
    gen = torch.Generator().manual_seed(3)
    draw = lambda r, c: torch.randint(-3, 4, (r, c), generator=gen).to(dtype)
    pairs = [(draw(m, k), draw(k, n)) for _ in range(2)]
    want = [a.double() @ b.double() for a, b in pairs]
    (a, b), (a2, b2) = [[t.cuda() for t in pair] for pair in pairs]
    c, c2 = torch.empty(m, n, device="cuda", dtype=out), torch.empty(m, n, device="cuda", dtype=out)
    torch.cuda.synchronize()
    call = lambda a, b, c, s: gemm(m, n, k, 1.0, a.data_ptr(), k, b.data_ptr(), n, 0.0, c.data_ptr(), n, stream=s)
    s = rt.stream_create()
    try:
        call(a2, b2, c2, s)
        with rt.Graph.capture(s) as graph:
            call(a, b, c, s)
        for _ in range(3):
            c.fill_(float("nan"))
            c2.fill_(float("nan"))
            torch.cuda.synchronize()
            graph.launch()
            call(a2, b2, c2, s)
            rt.stream_sync(s)
            assert torch.equal(c.double().cpu(), want[0]) and torch.equal(c2.double().cpu(), want[1])
        graph.destroy()
    finally:
        rt.stream_destroy(s)
