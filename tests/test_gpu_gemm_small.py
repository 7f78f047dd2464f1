"""The small GEMM class: the same bits as the 256-wide classes' summation order (the MN-major kernel on the transposed
bytes, which never takes it), at the edges of its tiles (32 x 64, 64 x 64, 128 x 64), partial K tiles, one to many K
tiles of its ring of stages, plans that split K (the splits' sums folded in their order), with bias and padded rows, and within the elementwise bound of the float64 product."""
import pytest
import torch

import gpic_fp8 as G
from parity import assert_elementwise

pytestmark = pytest.mark.gpu

# the last of each group lies just past the class's limit (256 CUs)
SHAPES = [(1, 16, 16), (31, 48, 128), (33, 80, 144), (32, 64, 256), (512, 1024, 384), (511, 1008, 400), (512, 1024, 1024),
          (1025, 1024, 512), (1024, 3072, 640), (4096, 768, 768), (4095, 784, 784), (4097, 1024, 1024), (2048, 1792, 1792),
          (4096, 1040, 1040), (2049, 3072, 1024),
          # split plans: even and uneven splits, a partial last K tile, K at and past the limit
          (300, 768, 3072), (512, 1024, 4096), (1111, 1152, 4608), (257, 1792, 7168), (2048, 768, 6000), (1000, 896, 8192),
          (1000, 896, 8208), (64, 64, 8192)]


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_small_gemm(dev, M, N, K, bias):
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    def operand(r):   # rows of a wider buffer, whose padding holds NaN bytes
        buf = torch.full((r, K + 16), 0x7f, dtype=torch.uint8, device=dev)
        buf[:, :K] = torch.randn(r, K, generator=g, device=dev).to(G.E4).view(torch.uint8)
        return buf.view(G.E4)[:, :K]
    a, b = operand(M), operand(N)
    sa, sb = torch.tensor([0.37], device=dev), torch.tensor([1.9], device=dev)
    bi = torch.randn(N, generator=g, device=dev).to(torch.bfloat16) if bias else None
    y = G.fp8_gemm(a, sa, b, sb, bi)
    if not bias:
        assert_elementwise(y, a, sa.item(), b, sb.item())
    # the MN-major kernel takes columns in multiples of 16
    m16 = M // 16 * 16
    if m16:
        t = lambda u: u.contiguous().view(torch.uint8).t().contiguous().view(G.E4)
        assert torch.equal(y[:m16], G.fp8_gemm_mn(t(a[:m16]), sa, t(b), sb, bi))


def _device_us(f):
    """The device time of f: the median of 9 replays of a graph of 20 launches."""
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


@pytest.mark.parametrize("M,N,K,most", [(16, 64, 8192, 1.15), (16, 1024, 8192, 1.15), (16, 1536, 6144, 1.15),
                                        (256, 3072, 8192, 1.15), (512, 6144, 4608, 0.95)])
def test_small_class_only_where_it_pays(dev, M, N, K, most):
    """Few rows of a long K, and small tiles that would stream a large B: no slower than the plan, whose time is taken from
    the MN-major layout's, which never has another class. (Measured ratios: 1.0 for split plans, 0.79 for the last, whose
    MN-major form is the slower one; with the small class 1.31-1.41, and 1.05.)"""
    g = torch.Generator(device=dev).manual_seed(K)
    a, b = (torch.randn(n, K, generator=g, device=dev).to(G.E4) for n in (M, N))
    at, bt = (t.view(torch.uint8).t().contiguous().view(G.E4) for t in (a, b))
    s = torch.ones(1, device=dev)
    assert _device_us(lambda: G.fp8_gemm(a, s, b, s)) < most * _device_us(lambda: G.fp8_gemm_mn(at, s, bt, s))
