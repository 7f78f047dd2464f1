"""The native host module against the general form of the same calls, bit for bit: linears of each recipe and the MLPs,
forward and backward, over the forms of input that either takes (rows 0, 1, odd; strided, misaligned and expanded
tensors; weight and bias types; autocast), and which of them the module takes at all."""
import pytest
import torch

import gpic_fp8 as G
from gpic_fp8 import _lib as L
from gpic_fp8 import fp8_native as F

pytestmark = pytest.mark.gpu
B16, F32, F16 = torch.bfloat16, torch.float32, torch.float16


def _tensor(g, shape, dtype, form):
    t = torch.randn(*shape, generator=g, device=g.device).to(dtype)
    if form == "strided":
        buf = torch.zeros(*shape[:-1], shape[-1] + 16, dtype=dtype, device=g.device)
        buf[..., :shape[-1]] = t
        return buf[..., :shape[-1]]
    if form == "misaligned":
        buf = torch.zeros(t.numel() + 1, dtype=dtype, device=g.device)
        buf[1:] = t.reshape(-1)
        return buf[1:].view(shape)
    if form == "columns":
        return t.transpose(-1, -2).contiguous().transpose(-1, -2)
    return t


def _grads(fn, ins, dy):
    ins = [None if t is None else t.detach().requires_grad_() for t in ins]
    y = fn(*ins)
    if not y.numel():
        return [y]
    return [y, *torch.autograd.grad(y, [t for t in ins if t is not None], dy if dy is not None else torch.ones_like(y))]


def _both(fn, ins, dy, monkeypatch):
    """fn's outputs and gradients with the host module and without it; the calls the module took."""
    took = []
    native = L.native

    def spy(name, *a):
        r = native(name, *a)
        took.append((name, r is not None))
        return r
    monkeypatch.setattr(L, "native", spy)
    a = _grads(fn, ins, dy)
    monkeypatch.setattr(L, "native", lambda *a: None)
    b = _grads(fn, ins, dy)
    monkeypatch.setattr(L, "native", native)
    assert len(a) == len(b)
    for s, t in zip(a, b):
        assert s.dtype == t.dtype and s.shape == t.shape and torch.equal(s, t)
    return took


@pytest.mark.parametrize("form", ["plain", "strided", "misaligned", "columns", "expanded dy"])
@pytest.mark.parametrize("rows", [1, 257])
@pytest.mark.parametrize("wdt", [F32, B16, F16])
@pytest.mark.parametrize("fn", [G.fp8_linear, G.fp8_linear_f8], ids=["native", "native3"])
def test_linear(dev, monkeypatch, fn, wdt, rows, form):
    g = torch.Generator(device=dev).manual_seed(rows)
    f = "plain" if form == "expanded dy" else form
    x = _tensor(g, (rows, 48), B16, f)
    w = _tensor(g, (272, 48), F32, f).to(wdt) if wdt == F16 else _tensor(g, (272, 48), wdt, f)
    b = _tensor(g, (272,), F32, "misaligned" if f == "misaligned" else "plain").to(wdt)
    dy = None if form == "expanded dy" else _tensor(g, (rows, 272), B16, f)
    took = _both(fn, [x, w, b], dy, monkeypatch)
    if form == "plain" and wdt != F16:
        assert took and all(ok for _, ok in took)
    _both(fn, [x.view(rows, 1, 48) if form == "plain" else x, w, None], None, monkeypatch)
    with torch.autocast("cuda", dtype=B16):
        _both(fn, [x.float(), w, b], dy, monkeypatch)


def test_no_rows(dev, monkeypatch):
    w = torch.randn(32, 16, device=dev)
    for fn in (G.fp8_linear, G.fp8_linear_f8):
        _both(fn, [torch.empty(0, 16, dtype=B16, device=dev), w, torch.randn(32, device=dev)], None, monkeypatch)


@pytest.mark.parametrize("fn", [G.fp8_mlp, G.fp8_mlp_f8], ids=["native2", "native3"])
def test_mlp(dev, monkeypatch, fn):
    g = torch.Generator(device=dev).manual_seed(5)
    x, w12, w3 = _tensor(g, (3, 67, 64), B16, "plain"), _tensor(g, (512, 64), F32, "plain"), _tensor(g, (64, 256), F32, "plain")
    took = _both(fn, [x, w12, w3], _tensor(g, (3, 67, 64), B16, "plain"), monkeypatch)
    assert {n for n, ok in took if ok} >= {"casts", "gemm"}


def test_errors_stay_errors(dev):
    x = torch.randn(8, 32, device=dev)
    with pytest.raises(ValueError):
        G.fp8_linear(x, torch.randn(16, 48, device=dev))       # K differs
    with pytest.raises(ValueError):
        G.fp8_linear_f8(x, torch.randn(24, 32, device=dev))    # N % 16
    with pytest.raises(RuntimeError, match="GPU only"):
        F.fp8_gemm(torch.zeros(16, 16).to(G.E4), torch.ones(1), torch.zeros(16, 16).to(G.E4), torch.ones(1))


@pytest.mark.parametrize("M,N,K", [(17, 48, 160), (2048, 1024, 1024), (512, 1024, 4096), (6592, 1024, 4096),
                                   (333, 3072, 1024), (33000, 272, 1024), (4096, 3072, 1040)])
def test_fp32_bias(dev, M, N, K):
    """An fp32 bias read by the GEMM (small, narrow, wide and split-K epilogues) gives the bits of its bf16 rounding."""
    g = torch.Generator(device=dev).manual_seed(M)
    a, b = (torch.randn(n, K, generator=g, device=dev).to(G.E4) for n in (M, N))
    s = torch.tensor([0.3], device=dev)
    bias = torch.randn(N, generator=g, device=dev)
    bias[0], bias[1], bias[2] = float("nan"), float("inf"), 1.00390625   # (the last: a tie)
    y, ref = G.fp8_gemm(a, s, b, s, bias), G.fp8_gemm(a, s, b, s, bias.to(B16))
    assert torch.equal(y.view(torch.int16), ref.view(torch.int16))
    buf = torch.zeros(N + 1, device=dev)
    buf[1:] = bias                                                       # not 16-byte aligned: the general form
    assert torch.equal(G.fp8_gemm(a, s, b, s, buf[1:]).view(torch.int16), ref.view(torch.int16))


def test_gemm_first_on_a_capturing_stream(dev, monkeypatch):
    """GEMMs captured on a stream that has no cast workspace make none, in a graph of their own; a later graph on that stream
    with a cast makes its own and gives the right bytes without the first one's replay."""
    monkeypatch.setattr(L, "_WORKSPACES", {})
    a, b, s = torch.randn(64, 128, device=dev).to(G.E4), torch.randn(32, 128, device=dev).to(G.E4), torch.ones(1, device=dev)
    c, w = F.fp8_gemm(a, s, b, s), F.fp8_wgrad(a, s, a, s, True)
    torch.cuda.synchronize()
    first, second, x = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph(), torch.randn(300, 80, device=dev).to(B16)
    with torch.cuda.graph(first):
        got = F.fp8_gemm(a, s, b, s), F.fp8_wgrad(a, s, a, s, True)
    assert not L._WORKSPACES
    with torch.cuda.graph(second, stream=torch.cuda.graph.default_capture_stream):
        q, sc = F.tcast(x)
    for k in range(3):
        x.mul_(0.5)
        second.replay()
        torch.cuda.synchronize()
        assert sc.item() == (x.abs().max().float().cpu() / torch.tensor(448.0)).item()   # (IEEE: on the GPU torch multiplies)
    first.replay()
    torch.cuda.synchronize()
    assert torch.equal(got[0], c) and torch.equal(got[1], w)


@pytest.mark.parametrize("name", ["casts", "gemm", "wgrad", "linear_fwd", "linear_bwd"])
def test_other_threads_run_during_a_call(dev, name):
    """The host module's calls release the GIL: a second Python thread, which with this switch interval never gets it unless
    the first gives it up, counts while the first does nothing but call the module."""
    import sys
    import threading
    import time
    index, stream = torch.cuda.current_device(), torch.cuda.current_stream().cuda_stream
    ws = L.cast_workspace(dev).data_ptr()
    x, w = torch.randn(64, 64, device=dev).to(B16), torch.randn(64, 64, device=dev)
    q, s = x.to(G.E4), torch.ones(1, device=dev)
    f = getattr(L.host(), name)
    args = {"casts": ([x, w], [F.FLAT, F.BOTH]), "gemm": (q, s, q, s, None), "wgrad": (q, s, q, s, True),
            "linear_fwd": (x, w, None, True), "linear_bwd": (x, q, s, q, s, True, True)}[name]
    count, running, stop = [0], threading.Event(), False

    def other():
        running.set()
        while not stop:
            count[0] += 1
            time.sleep(0)   # gives the GIL up
    t = threading.Thread(target=other)
    interval = sys.getswitchinterval()
    try:
        t.start()
        running.wait()
        sys.setswitchinterval(60.0)
        end = time.monotonic() + 0.1
        while time.monotonic() < end:   # (the other thread's wait that began under the old interval ends here)
            pass
        n, kept = count[0], []   # (results kept: freeing a tensor may give the GIL up as well)
        for _ in range(1000):
            kept.append(f(*args, index, ws, stream))
        got = count[0] - n
    finally:
        sys.setswitchinterval(interval)
        stop = True
        t.join()
    torch.cuda.synchronize()
    assert all(r is not None for r in kept) and got >= 500   # (several a call; none where the GIL is held)
