"""The attention form that cuts the keys between wavefronts and work-groups, against the oracle: key axes of less than a block,
of part of one and of more blocks than wavefronts, one query to more than a tile, keys cut between work-groups, rows whose
first finite score is in another wavefront's block, and a maximum that grows along the keys.

The bound is the one of the other forms: probabilities are rounded to bf16 (2^-9 of each term, 2e-2 of the largest result)."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import dev, rel_err_max

pytestmark = pytest.mark.gpu
TOL_BF16 = 2e-2


def run(rt, Q, K, V, causal=False, out_bf16=False):
    B, H, SQ, D = Q.shape
    q, k, v = (dev(t.contiguous().view(torch.int16).numpy().view(np.uint16)) for t in (Q, K, V))
    o = torch.full((B, H, SQ, D), float("nan"), device="cuda", dtype=torch.bfloat16 if out_bf16 else torch.float32)
    call = rt.attention_bf16_causal if causal else rt.attention_bf16
    call(B, H, SQ, K.shape[2], D, D ** -0.5, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), out_bf16=out_bf16)
    torch.cuda.synchronize()
    return o.float().cpu().numpy()


def expected(Q, K, V, causal=False):
    if not causal:
        return oracle.attention(*(t.contiguous().view(torch.int16).numpy().view(np.uint16) for t in (Q, K, V)))
    s = (Q.double() @ K.double().transpose(-1, -2).contiguous()) * Q.shape[-1] ** -0.5
    s = s.masked_fill(~torch.ones(s.shape[-2:], dtype=torch.bool).tril(), float("-inf"))
    return (torch.softmax(s, -1) @ V.double()).numpy()


def draw(seed, B, H, SQ, SKV, D):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(B, H, s, D, generator=g).bfloat16() for s in (SQ, SKV, SKV)]


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("B,H,SQ,SKV", [(1, 1, 1, 1), (1, 3, 1, 31), (2, 1, 33, 32), (1, 2, 32, 129), (1, 2, 65, 160), (1, 8, 5, 300)])
@pytest.mark.parametrize("causal", [False, True])
def test_edges_of_blocks_and_tiles(rt, monkeypatch, D, B, H, SQ, SKV, causal):
    monkeypatch.setenv("DOCC_ROCM_ATTENTION_Q", "32")
    Q, K, V = draw(SQ * 31 + SKV, B, H, SQ, SKV, D)
    for out_bf16 in (False, True):
        assert rel_err_max(run(rt, Q, K, V, causal, out_bf16), expected(Q, K, V, causal)) <= TOL_BF16


# no form forced: few heads and long key axes are cut between work-groups as well (2 to 64 of them), or there are few work-groups
@pytest.mark.parametrize("B,H,SQ,SKV,D,causal", [(1, 2, 1, 9001, 64, False), (1, 1, 3, 20000, 128, False), (2, 1, 40, 4100, 32, False),
                                                 (1, 1, 600, 600, 64, True), (1, 2, 1, 2048, 128, False)])
def test_parts_and_small_launches(rt, B, H, SQ, SKV, D, causal):
    Q, K, V = draw(SKV, B, H, SQ, SKV, D)
    for out_bf16 in (False, True):
        assert rel_err_max(run(rt, Q, K, V, causal, out_bf16), expected(Q, K, V, causal)) <= TOL_BF16


@pytest.mark.parametrize("SKV", [333, 6000])
def test_excluded_keys_and_growing_scores(rt, SKV):
    Q, K, V = draw(SKV, 1, 2, 3, SKV, 64)
    Q[..., 0] = Q[..., 0].abs() + 0.5
    K[0, 0, :SKV // 2, 0] = -float("inf")       # half of the blocks hold no finite score
    K[0, 1, :, 0] = (8.0 * (torch.arange(SKV) // 32 % 40)).bfloat16()      # e^(8 q0 / 8) from block to block
    O = run(rt, Q, K, V)
    assert np.isfinite(O).all() and rel_err_max(O, expected(Q, K, V)) <= TOL_BF16
    K[0, 1, :, 0] = -float("inf")               # nothing finite at all: NaN, as 0 / 0 gives
    O = run(rt, Q, K, V)
    assert np.isnan(O[0, 1]).all() and np.isfinite(O[0, 0]).all()


# whatever the form: the first 70 keys of a query score -inf, then come scores far below 0 (against a reference point of 0 every
# exponential is 0), or scores near 0 and behind them some that are larger by more than 2^40 (a move of the reference point from 0 up)
@pytest.mark.parametrize("form", ["32", "128", "256"])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_first_scores_that_are_not_finite(rt, monkeypatch, form, D, causal):
    monkeypatch.setenv("DOCC_ROCM_ATTENTION_Q", form)
    Q, K, V = draw(D, 1, 3, 300, 333, D)
    Q[..., 0] = 1
    K[0, :2, :70, 0] = -float("inf")
    K[0, 0, 70:, 0] = -256.0 * D ** 0.5
    K[0, 1, 200:, 0] = 64.0 * D ** 0.5
    O, want = run(rt, Q, K, V, causal), expected(Q, K, V, causal)
    first = 70 if causal else 0       # the queries before it see no finite score
    assert np.isnan(O[0, :2, :first]).all()
    for h in range(3):
        rows = slice(first if h < 2 else 0, None)
        assert rel_err_max(O[0, h, rows], want[0, h, rows]) <= TOL_BF16, h


def test_captured_call_cut_into_parts_replays(rt):
    Q, K, V = draw(5, 1, 2, 1, 9000, 64)
    q, k, v = Q.cuda(), K.cuda(), V.cuda()
    eager, o = torch.empty_like(q), torch.empty_like(q)
    args = (1, 2, 1, 9000, 64, 0.125, q.data_ptr(), k.data_ptr(), v.data_ptr())
    rt.attention_bf16(*args, eager.data_ptr(), out_bf16=True)
    torch.cuda.synchronize()
    s = rt.stream_create()
    try:
        with rt.Graph.capture(s) as graph:
            rt.attention_bf16(*args, o.data_ptr(), out_bf16=True, stream=s)
        for _ in range(3):
            o.fill_(float("nan"))
            torch.cuda.synchronize()
            graph.launch()
            rt.stream_sync(s)
            assert torch.equal(o, eager)
            rt.attention_bf16(*args, eager.data_ptr(), out_bf16=True)
            torch.cuda.synchronize()
        graph.destroy()
    finally:
        rt.stream_destroy(s)
