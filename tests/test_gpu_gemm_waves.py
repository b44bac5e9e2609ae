"""Products with K cut between the wavefronts of a work-group (csrc/kernels/gemm_waves.h), every tile, both orders of B: less than a piece of K, a part of one behind
many, ragged tiles, rows longer than K, C with a leading dimension of its own."""
import pytest
import torch

from docc_amd import runtime as rt

pytestmark = pytest.mark.gpu
ENTRY = {torch.float64: "docc_rocm_dgemm", torch.float32: "docc_rocm_sgemm"}


@pytest.fixture(autouse=True)
def _device():
    rt.init(0)


@pytest.mark.parametrize("tile", ["16", "32", "64", "1", None])
@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("dtype", list(ENTRY))
@pytest.mark.parametrize("m,n,k", [(1, 16, 8), (3, 24, 136), (16, 72, 1032), (33, 40, 72), (65, 136, 520), (130, 264, 264), (17, 16, 4104)])
def test_gemm_cut_between_wavefronts(monkeypatch, tile, trans_b, dtype, m, n, k):
    if tile:
        monkeypatch.setenv("DOCC_ROCM_GEMM_WAVES", tile)
    gen = torch.Generator().manual_seed(m * 31 + n)
    sum_type = torch.float64 if dtype == torch.float64 else torch.float32
    lda, ldc = k + 8, n + 3
    a = torch.randn(m, lda, generator=gen).to(dtype)
    b = torch.randn(*((n, k + 16) if trans_b else (k, n + 8)), generator=gen).to(dtype)
    a[:, k:] = float("nan")                       # behind the rows: not read, or dropped
    b[:, k if trans_b else n:] = float("inf")
    c = torch.randn(m, ldc, generator=gen).to(sum_type)
    bk = (b[:, :k].T if trans_b else b[:, :n]).double()
    exact, size = a[:, :k].double() @ bk, a[:, :k].double().abs() @ bk.abs()
    da, db = a.cuda(), b.cuda()
    for alpha, beta in ((1.0, 0.0), (0.5, -2.0)):
        got = c.clone()
        if beta == 0.0:
            got[:] = float("nan")
        keep = got[:, n:].clone()
        got = got.cuda()
        rt.call(ENTRY[dtype], 0, rt.NO_TRANS, rt.TRANS if trans_b else rt.NO_TRANS, m, n, k, alpha, da.data_ptr(), lda, db.data_ptr(), b.shape[1], beta, got.data_ptr(), ldc)
        torch.cuda.synchronize()
        got = got.cpu()
        ref = alpha * exact + (beta * c[:, :n].double() if beta else 0.0)
        # k products summed in the type of the sums (the oracle too, in fp64): at most k roundings of partial sums no larger than `size`, and the two of the store
        unit = 2.0 ** -53 if dtype == torch.float64 else 2.0 ** -24
        bound = unit * (2 * k * abs(alpha) * size + 4 * (ref.abs() + abs(beta) * c[:, :n].double().abs()))
        assert bool(((got[:, :n].double() - ref).abs() <= bound).all())
        assert torch.equal(got[:, n:].nan_to_num(7.0), keep.nan_to_num(7.0))
