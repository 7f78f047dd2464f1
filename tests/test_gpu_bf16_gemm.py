"""The bf16 wgrad (dy^T @ x): exact on small integers, and on normal data every element
within one bf16 rounding plus the fp32 accumulation's allowance of the float64 product, at the edges of the 256 x 256 and
256 x 128 tiles, partial K tiles of 64, K splits, one token, no tokens, and strided operands; fp32 outputs hold the bf16
ones' values; the e4m3 wgrad's fp32 output holds gpic_fp8_gemm_mn's values."""
import pytest
import torch

import gpic_fp8 as G
from gpic_fp8 import fp8_native as F

pytestmark = pytest.mark.gpu

# (tokens, rows, columns): one tile and its edges, narrow and wide plans, split K, partial K tiles
WGRAD = [(1, 16, 16), (63, 16, 272), (64, 256, 256), (65, 272, 144), (1000, 768, 3072), (13303, 896, 1792),
         (6592, 2048, 1024), (8200, 1040, 2064), (4096, 8192, 1024)]


def _data(g, ints, *shape):
    if ints:
        return torch.randint(-3, 4, shape, generator=g, device=g.device).to(torch.bfloat16)
    return torch.randn(*shape, generator=g, device=g.device).to(torch.bfloat16)


def _check(y, a, b, ints):
    ref = a.double() @ b.double()
    if ints:   # sums below 2^24: exact in fp32, one rounding
        assert torch.equal(y, ref.to(torch.bfloat16))
        return
    # half a bf16 ulp, and K fp32 roundings of the partial sums, each at most 2^-24 of the sum of magnitudes
    tol = ref.abs() * 2.0 ** -8 + (a.double().abs() @ b.double().abs()) * a.shape[1] * 2.0 ** -24 + 1e-30
    assert ((y.double() - ref).abs() <= tol).all()


def _strided(t, pad):
    buf = torch.full((t.shape[0], t.shape[1] + pad), float("nan"), dtype=t.dtype, device=t.device)
    buf[:, :t.shape[1]] = t
    return buf[:, :t.shape[1]]


@pytest.mark.parametrize("ints", [True, False])
@pytest.mark.parametrize("M,N,K", WGRAD)
def test_wgrad(dev, M, N, K, ints):
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    dy, x = _data(g, ints, M, N), _data(g, ints, M, K)
    y = F.bf16_wgrad(dy, x, False)
    _check(y, dy.t(), x, ints)
    y32 = F.bf16_wgrad(_strided(dy, 16), _strided(x, 8), True)
    assert y32.dtype == torch.float32 and torch.equal(y32, y.float())
    if M == 1:   # a single row's stride may be anything
        assert torch.equal(F.bf16_wgrad(dy.as_strided((1, N), (1, 1)), x.as_strided((1, K), (2, 1)), False), y)
    assert torch.equal(F.bf16_wgrad(dy.t().contiguous().t(), x, False), y)   # another stride order


def test_no_rows(dev):
    e = lambda *s: torch.empty(*s, dtype=torch.bfloat16, device=dev)
    for f32 in (False, True):
        assert not F.bf16_wgrad(e(0, 32), e(0, 64), f32).any()


@pytest.mark.parametrize("K,M,N", [(1, 16, 16), (127, 272, 144), (6592, 2048, 1024), (6592, 8192, 1024),
                                   (512, 4096, 4112), (4096, 1024, 1024)])
def test_e4m3_wgrad_f32(dev, K, M, N):
    g = torch.Generator(device=dev).manual_seed(K + M)
    a, b = (torch.randn(K, n, generator=g, device=dev).to(G.E4) for n in (M, N))
    sa, sb = torch.tensor([0.37], device=dev), torch.tensor([1.9], device=dev)
    y = F.fp8_wgrad(a, sa, b, sb, True)
    assert y.dtype == torch.float32 and torch.equal(y, G.fp8_gemm_mn(a, sa, b, sb).float())


def test_e4m3_wgrad_f32_scales_and_errors(dev):
    """The general form (strided operands) takes a scale as any one-element float tensor, as fp8_gemm_mn does, and refuses
    operands of different row counts."""
    a, b = (torch.randn(64, n + 16, device=dev).to(G.E4)[:, :n] for n in (32, 48))
    s = torch.tensor(0.5, dtype=torch.float64, device=dev)
    assert torch.equal(F.fp8_wgrad(a, s, b, s, True), G.fp8_gemm_mn(a, s, b, s).float())
    one = torch.ones(1, device=dev)
    for f32 in (False, True):
        with pytest.raises(ValueError):
            F.fp8_wgrad(a, one, b[:48], one, f32)
    with pytest.raises(ValueError):
        F.bf16_wgrad(a.to(torch.bfloat16), b[:48].to(torch.bfloat16), True)


@pytest.mark.parametrize("M,N,K,dt", [(1200, 1024, 1024, torch.bfloat16), (2048, 1280, 1280, torch.bfloat16),
                                      (2048, 1024, 1024, torch.float32), (512, 768, 768, torch.bfloat16),
                                      (4096, 1024, 1024, torch.bfloat16), (13303, 896, 1792, torch.float32)])
def test_the_faster_wgrad_is_taken(dev, M, N, K, dt):
    """A weight gradient of the bf16 backward: right either way, and its device time that of the faster of the kernel and
    the library's product (with its conversion for an fp32 weight)."""
    dy, x = torch.randn(M, N, device=dev).to(torch.bfloat16), torch.randn(M, K, device=dev).to(torch.bfloat16)

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
    with torch.no_grad():
        _check(F._wgrad16(dy, x, dt).to(torch.bfloat16), dy.t(), x, False)
        got = us(lambda: F._wgrad16(dy, x, dt))
        assert got < 1.1 * min(us(lambda: (dy.t() @ x).to(dt)), us(lambda: F.bf16_wgrad(dy, x, dt == torch.float32)))
