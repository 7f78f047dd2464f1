"""The work that a user of the FP8 linear path has it do, as timed cases: what a converted JiT-T2I model calls in one
layer of a training step (forward and backward) or of a sampler (forward only), through the package's public entry
points, and the two casts that a program calls by themselves.

listed() names the cases, draw(rng) gives further ones of the same ranges, prepare(case, seed) makes what a program
holds before the call, run(state) is one pass, work(case) the bytes and operations that a pass cannot do without,
tolerance(case) how far another correct implementation may be off, and exact(case, seed) the results with every sum
and every function in 64 bits, rounded only where the path's definition rounds (its bf16 tensors and e4m3 bytes).
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-gpic_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import gpic_fp8 as G  # noqa: E402

E4, BF, F32, F64 = torch.float8_e4m3fn, torch.bfloat16, torch.float32, torch.float64
EPS = 1e-6
WIDTHS = (768, 896, 1024, 1152, 1280, 1536, 1792)   # the model ladder's widths
MLP_KINDS = ("mlp_native", "mlp_native2", "mlp_native3", "norm_mlp")


def _case(name, kind, batch, tokens, width, out=0, weights="fp32", bias=False, outliers=False):
    """batch x tokens rows of `width` features; `out`: a linear's output features, an MLP's hidden size (4 x width
    when 0); weights: DDP keeps them in fp32 (widths below 1280), FSDP2 hands them over in bf16."""
    return {"name": name, "kind": kind, "batch": batch, "tokens": tokens, "width": width, "out": out or 4 * width,
            "weights": weights, "bias": bias, "outliers": outliers}


def listed():
    return [
        # A sampler's proj for one image with guidance (two rows of 256 tokens): the smallest call, latency and launches.
        _case("sample_proj_1img", "linear", 2, 256, 1024, out=1024, bias=True),
        # One FP8 linear forward, X [4096 x 768] . W [768 x 768], bf16: the smallest published configuration.
        _case("linear_4096x768", "linear", 16, 256, 768, out=768, weights="bf16"),
        # An image block's kv_y over the batch's caption tokens (128 captions, 51 each: an odd row count), training.
        _case("text_kv_train", "linear_f8", 128, 51, 1024, out=2048),
        # A text-refine block's SwiGLU MLP over 6592 caption tokens (128 x 51.5), training.
        _case("text_mlp_train", "mlp_native3", 64, 103, 1024),
        # A d12 image block's proj over the attention's own output, 16 heads of 64, with its bias, training.
        _case("d12_proj_heads_train", "heads_linear", 128, 256, 1024, out=1024, bias=True),
        # A d12 image block's first norm site with the qkv linear it feeds, training under DDP.
        _case("d12_norm_qkv_train", "norm_linear", 128, 256, 1024, out=3072),
        # A d12 image block's second norm site with the MLP it feeds, training under DDP: the larger part of its time.
        _case("d12_norm_mlp_train", "norm_mlp", 128, 256, 1024),
        # The SwiGLU MLP of a d10 block in the recipe "native" (FP8 forward, bf16 backward), training.
        _case("d10_mlp_native_train", "mlp_native", 128, 256, 768),
        # The SwiGLU MLP of a d11 block in the recipe "native2" (FP8 forward and dgrads), a ragged last batch of the
        # epoch with uncropped token counts, training.
        _case("d11_mlp_native2_ragged", "mlp_native2", 53, 251, 896),
        # The SwiGLU MLP of a d18 block on its micro-batch of 64 images, bf16 weights (FSDP2), activations with
        # outlier channels, training: the largest call.
        _case("d18_mlp_train", "mlp_native3", 64, 256, 1792, weights="bf16", outliers=True),
        # The activation cast alone, [32768 x 1024] bf16 with 1% outlier channels.
        _case("cast_32768x1024", "cast", 128, 256, 1024, out=0, weights="bf16", outliers=True),
        # A d12 block's four fp32 weights cast for the step (both layouts), as a program does before the block runs.
        _case("weight_casts_d12", "weight_casts", 1, 1, 1024),
    ]


def _cost(c):
    """A pass's time for keeping draws below the largest listed case: seconds at about half of this card's rates."""
    w = work(c)
    return w["flops"] / 1e15 + w["bytes"] / 2.5e12


def draw(rng):
    limit = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(("linear", "linear_f8", "heads_linear", "norm_linear", "norm_mlp", "mlp_native", "mlp_native2",
                           "mlp_native3", "cast", "weight_casts"))
        width = rng.choice(WIDTHS)
        tokens = rng.choice((256, 256, rng.randrange(16, 321), rng.randrange(16, 321)))
        rows = math.exp(rng.uniform(math.log(256), math.log(32768)))
        batch = max(1, round(rows / tokens))
        out = {"linear": rng.choice((width, 2 * width, 3 * width)), "linear_f8": rng.choice((width, 2 * width, 3 * width)),
               "heads_linear": width, "norm_linear": 3 * width}.get(kind, 4 * width)
        if kind == "heads_linear" and width % 64:
            continue
        c = _case("", kind, batch, tokens, width, out=out, weights=rng.choice(("fp32", "bf16")),
                  bias=kind == "heads_linear" or (kind == "linear" and out == width), outliers=rng.random() < 0.3)
        del c["name"]
        if _cost(c) <= limit:
            return c


# ------------------------------------------------------------------------------------------------ inputs

def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=g.device) * std


def _weight(g, c, n, k):
    return _randn(g, n, k, std=k ** -0.5).to(F32 if c["weights"] == "fp32" else BF)


def _acts(g, c, *shape):
    """N(0, 1) activations, 1% of the channels x50 where the case has outlier channels, rounded once to bf16."""
    x = _randn(g, *shape)
    if c["outliers"]:
        cols = torch.randperm(shape[-1], generator=g, device=g.device)[:max(1, round(0.01 * shape[-1]))]
        x[..., cols] *= 50.0
    return x.to(BF)


def prepare(case, seed):
    c = case
    g = torch.Generator(device="cuda").manual_seed(seed)
    B, N, C, O, kind = c["batch"], c["tokens"], c["width"], c["out"], c["kind"]
    s = {"case": c, "kind": kind}
    if kind == "weight_casts":   # qkv, proj, w12, w3
        s["ws"] = [_weight(g, c, n, k) for n, k in ((3 * C, C), (C, C), (2 * O, C), (C, O))]
        return s
    if kind == "heads_linear":   # the attention's output [B, H, N, 64]
        s["x"] = _acts(g, dict(c, outliers=False), B, C // 64, N, 64)
    else:
        s["x"] = _acts(g, c, B, N, C)
    if kind == "cast":
        return s
    if kind in MLP_KINDS:
        s["w12"], s["w3"] = _weight(g, c, 2 * O, C), _weight(g, c, C, O)
        s["dy"] = _randn(g, B, N, C, std=0.1).to(BF)
    else:
        s["w"] = _weight(g, c, O, C)
        if c["bias"]:
            s["b"] = _randn(g, O, std=0.02).to(s["w"].dtype)
        s["dy"] = _randn(g, B, N, O, std=0.1).to(BF)
    if kind in ("norm_linear", "norm_mlp"):
        s["wn"] = 1.0 + _randn(g, C, std=0.1)
        mod = _randn(g, B, 1, 6 * C, std=0.2).to(BF).chunk(6, dim=-1)   # adaLN's output and its views
        s["shift"], s["scale"] = mod[3], mod[4]
        if kind == "norm_mlp":
            s["gate"] = mod[2]
            s["a"] = _randn(g, B, N, C).to(BF)
            s["dxn"] = _randn(g, B, N, C, std=0.1).to(BF)
    if kind != "linear":
        for k in ("x", "a", "gate", "wn", "shift", "scale", "w", "b", "w12", "w3"):
            if k in s:
                s[k] = s[k].detach().requires_grad_(True)
    return s


# ------------------------------------------------------------------------------------------------ one pass

def run(state):
    s, kind = state, state["kind"]
    if kind == "cast":
        return G.tcast(s["x"])
    if kind == "weight_casts":
        return [t for cast in G.weight_casts(*s["ws"]) for t in cast]
    if kind == "linear":
        with torch.no_grad():
            return G.fp8_linear(s["x"], s["w"], s.get("b"))
    if kind == "norm_mlp":
        ins = [s[k] for k in ("x", "a", "gate", "wn", "shift", "scale", "w12", "w3")]
        xn, y = G.fp8_res_mod_rmsnorm_mlp(*ins[:6], EPS, *ins[6:])
        return [xn, y, *torch.autograd.grad((xn, y), ins, (s["dxn"], s["dy"]))]
    if kind == "norm_linear":
        ins = [s[k] for k in ("x", "wn", "shift", "scale", "w")]
        y = G.fp8_mod_rmsnorm_linear(*ins[:4], EPS, ins[4])
    elif kind in ("linear_f8", "heads_linear"):
        ins = [s[k] for k in ("x", "w", "b") if k in s]
        y = (G.fp8_linear_f8 if kind == "linear_f8" else G.fp8_heads_linear_f8)(*ins)
    else:
        ins = [s[k] for k in ("x", "w12", "w3")]
        if kind == "mlp_native":
            y = G.fp8_swiglu_w3(G.fp8_linear(ins[0], ins[1]), ins[2])
        else:
            y = (G.fp8_mlp if kind == "mlp_native2" else G.fp8_mlp_f8)(*ins)
    return [y, *torch.autograd.grad(y, ins, s["dy"])]


def work(case):
    c = case
    M, C, O, kind = c["batch"] * c["tokens"], c["width"], c["out"], c["kind"]
    wb = 4 if c["weights"] == "fp32" else 2
    if kind == "cast":
        return {"bytes": 3 * M * C + 4, "flops": 0}
    if kind == "weight_casts":
        n = 4 * C * C + 3 * C * O
        return {"bytes": (wb + 2) * n, "flops": 0}
    if kind == "linear":
        return {"bytes": 2 * M * (C + O) + wb * C * O, "flops": 2 * M * C * O}
    if kind in MLP_KINDS:   # x, dy in; y, dx out; w12, w3 in, their gradients out
        rows = 4 + (4 if kind == "norm_mlp" else 0)   # a, dxn in; x_new, da out
        return {"bytes": 2 * rows * M * C + 2 * wb * 3 * C * O, "flops": 18 * M * C * O}
    return {"bytes": 4 * M * (C + O) + 2 * wb * C * O, "flops": 6 * M * C * O}


def tolerance(case):
    """Bytes and scales are exact. The rest: about four times what the path differs from exact() by. A linear's outputs
    are one bf16 rounding of an fp32 sum (2.4e-4; 5e-4 with outlier channels, where one MFMA's sum of 128 products
    keeps fewer bits of the small ones); a norm site's bf16 parameter gradients also carry dh's roundings (8.6e-4). In
    an MLP a bf16 value that rounds the other way can move an e4m3 byte by one step in what follows (2e-3; 3.4e-3 with
    outlier channels); "max" is that step's effect on single elements (0.11; with outlier
    channels it is of the size of the values themselves, so only "rel" holds there)."""
    kind, out = case["kind"], case["outliers"]
    if kind in ("cast", "weight_casts"):
        return "exact"
    if kind in MLP_KINDS:
        return {"rel": 1.4e-2} if out else {"rel": 1e-2, "max": 0.4}
    if kind == "norm_linear":
        return {"rel": 3.5e-3, "max": 0.15}
    return {"rel": 2e-3 if out else 1e-3, "max": 0.06}


# ------------------------------------------------------------------------------------------------ 64 bits

def _b(t):
    """Rounded to bf16 where the path holds a bf16 tensor."""
    return t.to(BF).to(F64)


def _q(t):
    """The tensorwise e4m3 cast of t (exact in fp32): (bytes, dequantization scale), the path's rule in IEEE fp32."""
    f = t.to(F32)
    a = f.abs().amax().clamp_min(1e-12)
    k = torch.full_like(a, 448.0)
    return (f * (k / a)).clamp(-448.0, 448.0).to(E4), (a / k).reshape(1)


def _dq(t):
    """The values of t's e4m3 bytes without their scale, and the scale, in 64 bits."""
    q, s = _q(t)
    return q.to(F64), s.to(F64)


def _mm(a, b):
    """bf16(sa sb a @ b) of two (values, scale) pairs."""
    return _b((a[0] @ b[0]) * (a[1] * b[1]))


def _t(p):
    return p[0].t(), p[1]


def _swiglu(z):
    z1, z2 = z.chunk(2, dim=-1)
    return _b(_b(z1 * torch.sigmoid(z1)) * z2)


def _swiglu_bwd(z, da):
    z1, z2 = z.chunk(2, dim=-1)
    sg = torch.sigmoid(z1)
    return torch.cat([_b(da * z2 * (sg * (1 + z1 * (1 - sg)))), _b(da * _b(z1 * sg))], dim=-1)


def exact(case, seed):
    c, s = case, prepare(case, seed)
    kind, B, N, C = c["kind"], c["batch"], c["tokens"], c["width"]
    if kind == "cast":
        return _q(s["x"])
    if kind == "weight_casts":
        out = []
        for w in s["ws"]:
            q, d = _q(w)
            out += [q, q.view(torch.uint8).t().contiguous().view(E4), d]
        return out
    with torch.no_grad():
        wdt = F32 if c["weights"] == "fp32" else BF
        shape = s["x"].shape
        x = s["x"]
        if kind == "heads_linear":
            x = x.transpose(1, 2)
        x = x.reshape(-1, C).to(F64)
        dy = s["dy"].reshape(B * N, -1).to(F64) if "dy" in s else None

        def vec(k):   # a modulation chunk, one row per row of x
            return s[k].reshape(B, 1, C).to(F64).expand(B, N, C).reshape(-1, C)

        h = x
        if kind in ("norm_linear", "norm_mlp"):
            if kind == "norm_mlp":
                a, gate = s["a"].reshape(-1, C).to(F64), vec("gate")
                x = _b(x + gate * a)
            wn, sc = s["wn"].to(F64), vec("scale")
            rstd = torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)
            n = _b(wn * (x * rstd))
            h = _b(n * (1 + sc) + vec("shift"))

        if kind in MLP_KINDS:
            w12, w3 = s["w12"], s["w3"]
            hq, w12q, w3q, w3h = _dq(h), _dq(w12), _dq(w3), w3.to(BF).to(F64)
            z = _mm(hq, _t(w12q))
            aq = _dq(_swiglu(z))
            y = _mm(aq, _t(w3q))
            if kind in ("norm_mlp", "mlp_native3"):
                dyq = _dq(dy)
                dzq = _dq(_swiglu_bwd(z, _mm(dyq, w3q)))
                dh, dw12, dw3 = _mm(dzq, w12q), _mm(_t(dzq), hq), _mm(_t(dyq), aq)
            else:
                da = _mm(_dq(dy), w3q) if kind == "mlp_native2" else _b(dy @ w3h)
                dw3 = _b(dy.t() @ _b(aq[0] * aq[1]))
                dz = _swiglu_bwd(z, da)
                dh = _mm(_dq(dz), w12q) if kind == "mlp_native2" else _b(dz @ w12.to(BF).to(F64))
                dw12 = _b(dz.t() @ h)
            dws = [dw12.to(wdt), dw3.to(wdt)]
        else:
            hq, wq = _dq(h), _dq(s["w"])
            y = _mm(hq, _t(wq))
            if "b" in s:
                y = _b(y + s["b"].to(BF).to(F64))
            if kind == "linear":
                return y.view(B, N, -1)
            dyq = _dq(dy)
            dh, dws = _mm(dyq, wq), [_mm(_t(dyq), hq).to(wdt)]
            if "b" in s:
                dws.append(_b(dy.sum(0)).to(wdt))
        y = y.view(B, N, -1)
        if kind == "heads_linear":
            return [y, dh.view(B, N, C // 64, 64).transpose(1, 2), *dws]
        if kind not in ("norm_linear", "norm_mlp"):
            return [y, dh.view(shape), *dws]

        t = x * rstd
        dn = dh * (1 + sc)
        dt = dn * wn
        dx = rstd * (dt - t * (dt * t).mean(-1, keepdim=True))
        per = lambda v, like: v.view(B, N, C).sum(1).to(like.dtype).view(like.shape)
        dvec = [(dn * t).sum(0).to(F32), per(dh, s["shift"]), per(dh * n, s["scale"])]
        if kind == "norm_linear":
            return [y, _b(dx).view(shape), *dvec, *dws]
        dx = dx + s["dxn"].reshape(-1, C).to(F64)
        return [x.view(shape), y, _b(dx).view(shape), _b(dx * gate).view(shape), per(dx * a, s["gate"]), *dvec, *dws]
