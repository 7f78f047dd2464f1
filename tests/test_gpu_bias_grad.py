"""bias_grad: exact on small integers; on normal data every column within one bf16 rounding plus the fp32 sum's
allowance of the float64 sum, deterministic, at the edges of a workgroup's 256 columns and of its rows in flight, for
strided, transposed and expanded dy; fp32 output holds the bf16 one's values."""
import pytest
import torch

from gpic_fp8 import fp8_native as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N", [(0, 16), (1, 8), (7, 24), (32, 256), (33, 264), (1000, 768), (6528, 1024),
                                 (13303, 1792), (40000, 16), (5, 40000), (257, 12)])
def test_bias_grad(dev, M, N):
    g = torch.Generator(device=dev).manual_seed(M + N)
    i = torch.randint(-4, 5, (M, N), generator=g, device=dev).to(torch.bfloat16)
    assert torch.equal(F.bias_grad(i, False), i.double().sum(0).to(torch.bfloat16))   # |sums| < 2^24: exact in fp32
    dy = torch.randn(M, N, generator=g, device=dev).to(torch.bfloat16)
    db, ref = F.bias_grad(dy, False), dy.double().sum(0)
    tol = ref.abs() * 2.0 ** -8 + dy.double().abs().sum(0) * max(M, 1) * 2.0 ** -24
    assert ((db.double() - ref).abs() <= tol).all()
    db32 = F.bias_grad(dy, True)
    assert db32.dtype == torch.float32 and torch.equal(db32, db.float())
    buf = torch.full((M, N + 8), float("nan"), dtype=torch.bfloat16, device=dev)
    buf[:, :N] = dy
    assert torch.equal(F.bias_grad(buf[:, :N], False), db)
    assert torch.equal(F.bias_grad(dy.t().contiguous().t(), False), db)
    if M == 1:   # a single row's stride may be anything
        assert torch.equal(F.bias_grad(dy.as_strided((1, N), (1, 1)), False), db)
    one = torch.ones((), dtype=torch.bfloat16, device=dev).expand(M, N)   # what sum().backward() hands over
    assert torch.equal(F.bias_grad(one, True), torch.full((N,), float(M), device=dev).to(torch.bfloat16).float())


def test_bias_grad_nan(dev):
    dy = torch.ones(70, 512, dtype=torch.bfloat16, device=dev)
    dy[69, 3], dy[0, 4], dy[1, 4] = float("nan"), float("inf"), float("-inf")
    db = F.bias_grad(dy, False)
    assert db[3].isnan() and db[4].isnan() and (db.nan_to_num(70.0) == 70).all()


@pytest.mark.parametrize("M,N", [(1, 8), (7, 456), (8, 2144), (16, 480)])
def test_bias_grad_of_few_rows_is_one_launch(dev, M, N):
    """Up to 32 rows a bf16 bias's gradient takes no longer than torch's sum, which is one launch too."""
    dy = torch.randn(M, N, device=dev).to(torch.bfloat16)

    def us(f):   # the median of 9 replays of a graph of 20 launches
        f()
        torch.cuda.synchronize()
        graph, times = torch.cuda.CUDAGraph(), []
        with torch.cuda.graph(graph):
            for _ in range(20):
                f()
        for _ in range(9):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            graph.replay()
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end) * 1e3 / 20)
        return sorted(times)[4]
    assert not F.bias_grad(-torch.zeros_like(dy), False).signbit().any()   # (-0 sums to +0, as the partials' sum gives)
    assert us(lambda: F.bias_grad(dy, False)) < 1.12 * us(lambda: dy.sum(0))
