"""The MN-major GEMMs (e4m3 and bf16) over any number of K rows: rows past the last, partial K tile -- which lie in the
same buffer here, filled with NaN -- take no part, for both tile widths, K splits and the columns' edges. The results are
those of the operands padded with zero rows to whole K tiles, bit for bit."""
import pytest
import torch

import gpic_fp8 as G
from gpic_fp8 import fp8_native as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N", [(16, 16), (272, 144), (1024, 1024), (2048, 1040), (8192, 1024)])
@pytest.mark.parametrize("K", [1, 63, 64, 65, 127, 129, 1000, 6592, 6599])
def test_rows_past_k(dev, K, M, N):
    g = torch.Generator(device=dev).manual_seed(K + M)
    full = (K + 127) // 128 * 128
    s = torch.tensor([0.5], device=dev)

    def operands(dtype):
        ops = []
        for n in (M, N):
            t = torch.randn(K, n, generator=g, device=dev).to(dtype)
            bits = torch.uint8 if dtype == G.E4 else torch.int16
            nan = torch.full((full + 128, n), 0x7f if dtype == G.E4 else 0x7fff, dtype=bits, device=dev)
            zero = torch.zeros(full, n, dtype=bits, device=dev)
            nan[:K], zero[:K] = t.view(bits), t.view(bits)
            ops.append((nan.view(dtype)[:K], zero.view(dtype)))
        return ops
    (a, az), (b, bz) = operands(G.E4)
    for f32 in (False, True):
        assert torch.equal(F.fp8_wgrad(a, s, b, s, f32), F.fp8_wgrad(az, s, bz, s, f32))
    (a, az), (b, bz) = operands(torch.bfloat16)
    assert torch.equal(F.bf16_wgrad(a, b, False), F.bf16_wgrad(az, bz, False))


@pytest.mark.parametrize("K,ld", [(1, 1 << 26), (15, 1 << 26), (15, (1 << 26) + 16), (60, 1 << 25), (63, (1 << 24) + 16),
                                  (63, 1 << 24)])
def test_long_row_strides(dev, K, ld):
    """Column slices of very wide tensors, whose row strides times the rows of a whole K tile pass 2^31 and 2^32 bytes: the
    K rows past the last take no part, and the results are those of contiguous copies, bit for bit."""
    g = torch.Generator(device=dev).manual_seed(K)
    s = torch.tensor([0.5], device=dev)
    M, N = 272, 48
    for dtype in (G.E4, torch.bfloat16):
        bits = torch.uint8 if dtype == G.E4 else torch.int16
        ops = []
        for n in (M, N):
            buf = torch.full((K, ld), 0x7f if dtype == G.E4 else 0x7fff, dtype=bits, device=dev)   # NaN beside the slice
            t = torch.randn(K, n, generator=g, device=dev).to(dtype)
            buf[:, :n] = t.view(bits)
            ops.append((buf.view(dtype)[:, :n], t))
        (a, ac), (b, bc) = ops
        assert a.stride(0) == ld and b.stride(0) == ld
        if dtype == G.E4:
            assert torch.equal(G.fp8_gemm_mn(a, s, b, s), G.fp8_gemm_mn(ac, s, bc, s))
            assert torch.equal(G.fp8_gemm_mn(ac, s, b, s), G.fp8_gemm_mn(ac, s, bc, s))
            assert torch.equal(F.fp8_wgrad(a, s, b, s, True), F.fp8_wgrad(ac, s, bc, s, True))
        elif 2 * K * ld < 2 ** 31:   # (past it, another route)
            for f32 in (False, True):
                assert torch.equal(F.bf16_wgrad(a, b, f32), F.bf16_wgrad(ac, bc, f32))
        del ops, a, b, buf
