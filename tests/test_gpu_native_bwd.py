"""The one-pass elementwise kernels of the bf16 backwards (recipes native, native2): swiglu_dz gives swiglu_bwd's dz bit
for bit, dequant gives torch's (q.float() * s).to(bfloat16) bit for bit, at sizes around a workgroup's share, with
strided rows, NaN and infinities; and _SwiGLUw3's backward agrees with its recorded (create_graph) form, which is the
torch expression, within the sigmoid's two fp32 ulp (one bf16 ulp of dz)."""
import pytest
import torch

import gpic_fp8 as G
from gpic_fp8 import fp8_native as F

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.contiguous().view(torch.int16)


@pytest.mark.parametrize("M,H,pad", [(1, 8, 0), (3, 8, 16), (511, 8, 0), (513, 24, 8), (64, 4096, 0), (1023, 1032, 8),
                                     (2049, 3584, 0)])
def test_swiglu_dz(dev, M, H, pad):
    g = torch.Generator(device=dev).manual_seed(M + H)
    z = torch.randn(M, 2 * H + pad, generator=g, device=dev).mul_(4).to(torch.bfloat16)[:, :2 * H]
    da = torch.randn(M, H + pad, generator=g, device=dev).to(torch.bfloat16)[:, :H]
    z[0, 0], z[M - 1, H], da[0, H - 1] = float("inf"), float("nan"), float("-inf")
    z[0, 1], z[0, 2] = 0.0, -1e-30
    dz = F.swiglu_dz(z, da)
    assert torch.equal(_bits(dz), _bits(G.swiglu_bwd(z, da)[0]))


def test_swiglu_dz_empty(dev):
    z = torch.empty(0, 64, dtype=torch.bfloat16, device=dev)
    assert F.swiglu_dz(z, torch.empty(0, 32, dtype=torch.bfloat16, device=dev)).shape == (0, 64)


@pytest.mark.parametrize("n", [0, 1, 15, 16, 17, 256, 16 * 256 * 4 + 5, 1 << 20, 3 * (1 << 23) + 3])
def test_dequant(dev, n):
    q = (torch.arange(n, device=dev) % 256).to(torch.uint8).view(G.E4)
    s = torch.tensor([0.0123456], device=dev)
    y = F.dequant(q, s)
    ref = (q.float() * s).to(torch.bfloat16)
    nan = ref.isnan()
    assert torch.equal(y.isnan(), nan) and torch.equal(_bits(y)[~nan], _bits(ref)[~nan])


def test_native_backward_matches_its_recorded_form(dev):
    g = torch.Generator(device=dev).manual_seed(3)
    z = torch.randn(3, 100, 2 * 96, generator=g, device=dev).to(torch.bfloat16).requires_grad_()
    w3 = (torch.randn(64, 96, generator=g, device=dev) / 10).requires_grad_()
    dy = torch.randn(3, 100, 64, generator=g, device=dev).to(torch.bfloat16).requires_grad_()
    y = G.fp8_swiglu_w3(z, w3)
    a = torch.autograd.grad(y, (z, w3), dy, retain_graph=True)
    b = torch.autograd.grad(y, (z, w3), dy, create_graph=True)
    assert torch.equal(a[1], b[1])
    d = (a[0].float() - b[0].float()).abs()
    assert (d <= 2.0 ** -7 * b[0].float().abs() + 1e-30).all()   # one bf16 ulp
    # the recorded form stays differentiable (dz is linear in dy and w3)
    for h in torch.autograd.grad(b[0].float().pow(2).sum(), (dy, w3)):
        assert h.abs().sum() > 0
