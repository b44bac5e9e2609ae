"""Launchers on a stream that another library captures (torch's graphs): the calls that would take a block of the runtime's cache run in a form
without one, and the graph's replays, with the program's own calls between them, give what the eager call gives."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def whole(*shape, dtype=torch.float32, seed=0):
    # small whole numbers: every sum is exact in fp32, whatever form adds it up
    return torch.randint(-3, 4, shape, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()


def packed_gemm(rt):
    a, b, c = whole(260, 333, dtype=torch.bfloat16), whole(333, 129, dtype=torch.bfloat16), torch.empty(260, 129, device="cuda")
    return lambda s: rt.bf16gemm_f32(260, 129, 333, 1.0, a.data_ptr(), 333, b.data_ptr(), 129, 0.0, c.data_ptr(), 129, stream=s), c


def cut_gemm(rt):
    a, b, c = whole(512, 8192), whole(8192, 1024), torch.empty(512, 1024, device="cuda")
    return lambda s: rt.sgemm(512, 1024, 8192, 1.0, a.data_ptr(), 8192, b.data_ptr(), 1024, 0.0, c.data_ptr(), 1024, stream=s), c


def few_columns(rt):
    a, b, c = whole(2048, 512), whole(512, 9), torch.empty(2048, 9, device="cuda")
    return lambda s: rt.sgemm(2048, 9, 512, 1.0, a.data_ptr(), 512, b.data_ptr(), 9, 0.0, c.data_ptr(), 9, stream=s), c


def cut_convolution(rt):
    x, w, y = whole(1, 256, 14, 14), whole(256, 256, 3, 3), torch.empty(1, 256, 14, 14, device="cuda")
    return lambda s: rt.conv2d_f32(1, 256, 14, 14, 256, 3, 3, (1, 1), (1, 1), (1, 1), x.data_ptr(), w.data_ptr(), 0, y.data_ptr(), stream=s), y


def cut_attention(rt):
    # equal scores: the mean of 8192 whole numbers, a multiple of 2^-13, exact in fp32
    q, k, v = torch.zeros(1, 2, 1, 64, device="cuda").bfloat16(), whole(1, 2, 8192, 64, dtype=torch.bfloat16), whole(1, 2, 8192, 64, dtype=torch.bfloat16, seed=1)
    o = torch.empty(1, 2, 1, 64, device="cuda")
    return lambda s: rt.attention_bf16(1, 2, 1, 8192, 64, 0.125, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), stream=s), o


@pytest.mark.parametrize("case", [packed_gemm, cut_gemm, few_columns, cut_convolution, cut_attention])
def test_a_captured_call_replays(rt, case):
    call, out = case(rt)
    call(0)                                  # kernels are looked up, and the form with a block runs
    torch.cuda.synchronize()
    want = out.clone()
    cached = rt.pool_stats()
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=stream):
        call(stream.cuda_stream)
    assert rt.pool_stats() == cached         # nothing was taken or given back
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        call(0)
        torch.cuda.synchronize()
        assert torch.equal(out, want)
