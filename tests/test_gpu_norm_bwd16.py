"""The norm site's backward with bf16 modulation gradients: the fp32 form's outputs, with d_shift, d_scale and d_gate
rounded once to bf16."""
import pytest
import torch

from gpic_fp8 import norm as NM

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,N,C,res,dxn", [(1, 1, 4, False, False), (3, 65, 256, True, True), (2, 130, 896, True, False),
                                           (5, 64, 1792, False, False), (0, 7, 64, True, True)])
def test_bwd_bf16_vectors(dev, B, N, C, res, dxn):
    g = torch.Generator(device=dev).manual_seed(C)
    r = lambda *s: torch.randn(*s, generator=g, device=dev).to(torch.bfloat16)
    a, gate = (r(B, N, C), r(B, 1, C)) if res else (None, None)
    args = (r(B, N, C), r(B, N, C) if dxn else None, r(B, N, C), a, gate, 1 + r(C).float(), r(B, 1, C),
            torch.rand(B * N, generator=g, device=dev) + 0.5)
    ref, got = NM.res_mod_rmsnorm_bwd_k(*args), NM.res_mod_rmsnorm_bwd16(*args)
    for i, (s, t) in enumerate(zip(ref, got)):
        want = s.to(torch.bfloat16) if i in (2, 4, 5) else s
        assert t.dtype == want.dtype and torch.equal(t, want), i
