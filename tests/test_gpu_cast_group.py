"""cast_group: every tensor's bytes and scale equal tcast's / tcast_t's bit for bit, for each set of kinds that shares a
launch and for sets, sizes and settings that take the per-tensor calls, with a zero wait bound (every partial computed
by the waiting workgroup), NaN and infinities, odd sizes, and as a captured graph replayed."""
import pytest
import torch

import gpic_fp8 as G
from gpic_fp8 import _lib as L
from gpic_fp8 import fp8_native as F

pytestmark = pytest.mark.gpu
B16, F32 = torch.bfloat16, torch.float32
FL, BO, TR = F.FLAT, F.BOTH, F.TRANSPOSED

# (shape, dtype, kind) of each tensor
SETS = [
    [((1, 8), B16, FL), ((16, 16), F32, BO)],                                        # one workgroup each
    [((512, 1024), B16, FL), ((1024, 1024), F32, BO)],
    [((4096, 768), B16, FL), ((768, 768), B16, FL)],
    [((4095, 777), B16, FL), ((300, 333), F32, FL)],                                 # tails of both
    [((6528, 1024), B16, FL), ((2048, 1024), B16, BO)],
    [((6592, 1024), B16, FL), ((8192, 1024), F32, BO), ((1024, 4096), F32, BO)],
    [((13303, 896), B16, FL), ((7168, 896), F32, TR), ((896, 3584), F32, TR)],       # qt alone; 16 words a thread
    [((8192, 1024), F32, BO), ((1024, 4096), F32, BO), ((1000, 272), F32, TR)],
    [((9216, 1152), F32, BO), ((1152, 4608), F32, BO)],                              # past 1024 workgroups: per tensor
    [((32768, 1024), B16, FL), ((1024, 1024), F32, BO)],                             # x fills the device: per tensor
    [((64, 64), F32, FL), ((64, 64), B16, BO)],                                      # a set with no instance
    [((0, 64), B16, FL), ((64, 64), B16, BO)],                                       # an empty tensor
    [((37,), B16, FL)] * 9,                                                          # more than a launch takes
]


def _bytes(t):
    return t.contiguous().view(torch.uint8)


def _same(xs, kinds, out):
    for i, (x, k) in enumerate(zip(xs, kinds)):
        q, qt, s = out[3 * i:3 * i + 3]
        if k == FL:
            q0, s0 = G.tcast(x)
            assert qt.numel() == 0
        else:
            q0, qt0, s0 = G.tcast_t(x)
            assert torch.equal(_bytes(qt), _bytes(qt0))
        assert torch.equal(s, s0)
        if k == TR:
            assert q.numel() == 0
        else:
            assert q.shape == x.shape and torch.equal(_bytes(q), _bytes(q0))


@pytest.fixture
def knob():
    yield
    L.set_single_pass(True, -1)


@pytest.mark.parametrize("wait", [-1, 0, None])
@pytest.mark.parametrize("tensors", SETS, ids=lambda s: "+".join("x".join(map(str, t[0])) for t in s[:3]))
def test_cast_group(dev, knob, tensors, wait):
    g = torch.Generator(device=dev).manual_seed(7)
    xs = [(torch.randn(*sh, generator=g, device=dev) * 10.0 ** (i % 4 - 1)).to(dt) for i, (sh, dt, _) in enumerate(tensors)]
    kinds = [k for _, _, k in tensors]
    if xs[0].numel() > 8:
        xs[0].view(-1)[-1] = float("nan")      # leaves that tensor's amax, and no other's, unchanged
    if len(xs) > 2:
        xs[1].view(-1)[3] = float("inf")
    L.set_single_pass(wait is not None, -1 if wait is None else wait)
    out = F.cast_group(xs, kinds)
    L.set_single_pass(True, -1)
    _same(xs, kinds, out)


def test_cast_group_in_a_graph(dev):
    x, w = torch.randn(512, 256, device=dev).to(B16), torch.randn(256, 256, device=dev)
    F.cast_group([x, w], [FL, BO])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = F.cast_group([x, w], [FL, BO])
    for k in range(4):
        x.copy_(torch.randn(512, 256, device=dev).to(B16) * 10.0 ** k)
        w.mul_(0.3)
        graph.replay()
        torch.cuda.synchronize()
        _same([x, w], [FL, BO], out)


def test_cast_group_errors(dev):
    x = torch.randn(16, 24, device=dev)
    with pytest.raises(ValueError):
        F.cast_group([x, x], [FL, BO])
