"""The work a program that serves sys1's models has the projection path do,
as timed cases: single projections through their modules, a block of layers
and a whole encoder stack through ProjectionStack.

A case is a dict of plain values.  `kind` names the entry point:
  linear  sys1_amd.linear.Linear       (bias, GELU and residual as options)
  gated   sys1_amd.linear.GatedLinear  (GeGLU / SwiGLU)
  norm    sys1_amd.norm.NormLinear     (LayerNorm / RMSNorm fused, gated or not)
  rope    sys1_amd.rope.RopeQkvLinear
  conv    sys1_amd.deltanet.InProjConv (causal conv + SiLU, RMSNorm optional)
  stack   sys1_amd.stacks.ProjectionStack (ModernBERT layers, norms fused)
M is the packed token count, K the input width, N the weight rows (both
halves of a gated weight).  Widths are those of stacks.CONFIGS.
"""
from __future__ import annotations

import math

import torch

from sys1_amd.batching import draw_lengths, positions

DEV = "cuda:0"

# (name, K, N) of the projections of the models that stacks.CONFIGS lists.
ENCODER = {
    "base": (768, 1152, 12),     # hidden, intermediate, heads of 64
    "large": (1024, 2624, 16),
}
# hidden, intermediate, in_proj width, conv channels, out_proj input, q|k|v width
DECODER = {
    "small": (2048, 6144, 12320, 8192, 4096, 4608),
    "27b": (5120, 17408, 16480, 10240, 6144, 14336),
}
VISION = (1152, 4304)

# Largest work of a drawn case: that of the largest listed one.
MAX_FLOPS = 2.0 * 4096 * 34816 * 5120


def listed():
    return [
        # The Laya scorer's first layer on the pooled rows of a few requests:
        # the smallest call of the path, a launch and a latency.
        dict(name="scorer_m16", kind="linear", M=16, K=768, N=768, bias=True, act="erf", residual=False,
             blocked=False),
        # One short request through an encoder: Wqkv with RoPE.
        dict(name="base_rope_qkv_m61", kind="rope", M=61, K=768, heads=12),
        # Two encoder layers of a small batch, norms fused: eight dependent
        # launches, where launch gaps and latency count.
        dict(name="large_layers_m64", kind="stack", M=64, hidden=1024, inter=2624, layers=2, blocked=True),
        # A middle batch: the MLP's output projection and its residual.
        dict(name="large_mlp_wo_m1024", kind="linear", M=1024, K=2624, N=1024, bias=False, act="", residual=True,
             blocked=False),
        # The encoder's ordinary batch (ragged, packed up to 8192 tokens).
        dict(name="base_wqkv_m8109", kind="linear", M=8109, K=768, N=2304, bias=False, act="", residual=False,
             blocked=False),
        dict(name="base_ln_wi_geglu_m8109", kind="norm", M=8109, K=768, N=2304, norm="layer", act="gelu",
             blocked=False),
        # Prefill of the hybrid decoder: RMSNorm + in_proj + causal conv.
        dict(name="small_in_proj_conv_m8192", kind="conv", M=8192, K=2048, N=12320, C=8192, norm=True),
        # Decode steps of eight sequences on the 27B widths: a weight stream.
        dict(name="27b_rms_qkv_m8", kind="norm", M=8, K=5120, N=14336, norm="rms", act="", blocked=True),
        # A short prefill there: deep K, residual.
        dict(name="27b_down_m128", kind="linear", M=128, K=17408, N=5120, bias=False, act="", residual=True,
             blocked=True),
        # The largest projection: gate/up of a long prefill.
        dict(name="27b_rms_gate_up_m4096", kind="norm", M=4096, K=5120, N=34816, norm="rms", act="silu",
             blocked=True),
        # Patch rows of an image through the vision tower's fc1, an odd count.
        dict(name="vision_fc1_m3001", kind="linear", M=3001, K=1152, N=4304, bias=True, act="tanh", residual=False,
             blocked=False),
        # The whole encoder: every projection of 22 layers with its norms.
        dict(name="base_stack_m8109", kind="stack", M=8109, hidden=768, inter=1152, layers=22, blocked=True),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a model width or a generic odd one, tokens over 1..16384
    on a logarithmic scale, every option of its entry point."""
    while True:
        M = max(1, min(16384, _log_uniform(rng, 1, 16384)))
        blocked = rng.random() < 0.5
        kind = rng.choice(["linear", "linear", "gated", "norm", "norm", "rope", "conv", "stack"])
        enc = ENCODER[rng.choice(sorted(ENCODER))]
        dec = DECODER[rng.choice(sorted(DECODER))]
        if kind == "rope":
            c = dict(kind=kind, M=M, K=enc[0], heads=enc[2])
        elif kind == "conv":
            c = dict(kind=kind, M=M, K=dec[0], N=dec[2], C=dec[3], norm=rng.random() < 0.7)
        elif kind == "stack":
            c = dict(kind=kind, M=M, hidden=enc[0], inter=enc[1], layers=rng.randint(1, 4), blocked=blocked)
        elif kind == "gated":
            if rng.random() < 0.5:
                c = dict(kind=kind, M=M, K=enc[0], N=2 * enc[1], act="gelu", blocked=blocked)
            else:
                c = dict(kind=kind, M=M, K=dec[0], N=2 * dec[1], act="silu", blocked=blocked)
        elif kind == "norm":
            c = rng.choice([
                dict(K=enc[0], N=3 * enc[0], norm="layer", act=""),
                dict(K=enc[0], N=2 * enc[1], norm="layer", act="gelu"),
                dict(K=dec[0], N=dec[5], norm="rms", act=""),
                dict(K=dec[0], N=2 * dec[1], norm="rms", act="silu"),
            ])
            c = dict(kind=kind, M=M, blocked=blocked, **c)
        else:
            H, I = VISION
            K, N = rng.choice([
                (enc[0], 3 * enc[0]), (enc[0], enc[0]), (enc[1], enc[0]),
                (dec[0], dec[5]), (dec[4], dec[0]), (dec[1], dec[0]),
                (H, 3 * H), (H, I), (I, H),
                (8 * rng.randint(8, 400), rng.randint(33, 5000)),  # a generic odd projection
            ])
            bias = K in VISION or rng.random() < 0.3
            act = rng.choice(["", "erf", "tanh"]) if bias else ""
            c = dict(kind=kind, M=M, K=K, N=N, bias=bias, act=act, residual=not act and rng.random() < 0.5,
                     blocked=blocked)
        if work(c)["flops"] <= MAX_FLOPS:
            return c


def _stack_weights(c):
    H, I = c["hidden"], c["inter"]
    return [(3 * H, H), (H, H), (2 * I, H), (H, I)]


def work(c):
    M = c["M"]
    if c["kind"] == "stack":
        n = sum(a * b for a, b in _stack_weights(c)) * c["layers"]
        # the weights, the input and the result; what passes between the
        # projections of a layer stays on the chip at best
        return {"flops": 2.0 * M * n, "bytes": 2.0 * (n + 2 * M * c["hidden"])}
    K = c["K"]
    N = 3 * 64 * c["heads"] if c["kind"] == "rope" else c["N"]
    gated = c["kind"] == "gated" or (c["kind"] == "norm" and c["act"])
    out = N // 2 if gated else N
    b = 2.0 * (M * K + N * K + M * out)
    if c.get("residual"):
        b += 2.0 * M * out
    if c.get("bias"):
        b += 2.0 * N
    if c["kind"] == "conv":
        b += 2.0 * 4 * c["C"] + 4.0 * M
    if c["kind"] == "rope":
        b += 4.0 * M + 2 * 4.0 * 32 * min(M, 8192)
    return {"flops": 2.0 * M * N * K, "bytes": b}


def tolerance(c):
    # One bf16 rounding of the result is 1.7e-3 of it (2-norm); each further
    # rounded step of an epilogue adds its share.  Measured against exact():
    # 1.7e-3 plain, 2.0-2.6e-3 with one more step, 3.3e-3 with bias and GELU,
    # 4.3e-3 gated after a folded norm weight; 4e-3 over two encoder layers
    # and 1.2e-2 over 22.
    if c["kind"] == "stack":
        return {"rel": 0.016 if c["layers"] <= 4 else 0.03, "max": 0.5}
    gated = c["kind"] == "gated" or (c["kind"] == "norm" and c["act"])
    return {"rel": 0.016 if gated or c.get("act") else 0.01, "max": 0.1}


def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed(1_000_003 * int(seed) + stream)
    return g


def _randn(seed, stream, *shape, std=1.0):
    return torch.randn(*shape, generator=_gen(seed, stream), device=DEV) * std


def _hidden(seed, M, K):
    """A residual stream before its norm: unit noise, an offset per row and a
    few channels that run large, as trained models show."""
    x = _randn(seed, 1, M, K) + 0.2 * _randn(seed, 2, M, 1)
    loud = torch.randperm(K, generator=_gen(seed, 3), device=DEV)[:max(1, K // 256)]
    x[:, loud] *= 8.0
    return x.to(torch.bfloat16)


def _lengths(seed, M):
    hi = max(1, min(512, M))
    return draw_lengths(int(seed), max(1, min(16, hi)), hi, M, exact=True)


def _inputs(c, seed):
    """Every tensor of the case, made from the seed (bf16 on the GPU): the
    same for prepare() and exact()."""
    M, k = c["M"], c["kind"]
    t = {}
    if k == "stack":
        t["x"] = _hidden(seed, M, c["hidden"])
        t["w"] = [[_randn(seed, 100 + 10 * i + j, n, kk, std=0.02).to(torch.bfloat16)
                   for j, (n, kk) in enumerate(_stack_weights(c))] for i in range(c["layers"])]
        t["g"] = [[1.0 + 0.1 * _randn(seed, 5000 + 10 * i, c["hidden"]) if i else None, None,
                   1.0 + 0.1 * _randn(seed, 5001 + 10 * i, c["hidden"]), None] for i in range(c["layers"])]
        return t
    K = c["K"]
    N = 3 * 64 * c["heads"] if k == "rope" else c["N"]
    normed = k == "norm" or (k == "conv" and c["norm"])
    t["x"] = _hidden(seed, M, K) if normed else _randn(seed, 1, M, K).to(torch.bfloat16)
    t["w"] = _randn(seed, 4, N, K, std=0.02).to(torch.bfloat16)
    if k == "norm":
        t["g"] = 0.1 * _randn(seed, 5, K) + (1.0 if c["norm"] == "layer" else 0.0)
    if k == "conv":
        t["g"] = 0.1 * _randn(seed, 5, K) if c["norm"] else None
        t["cw"] = _randn(seed, 6, c["C"], 4, std=0.5).to(torch.bfloat16)
    if c.get("bias"):
        t["b"] = _randn(seed, 7, N, std=0.1).to(torch.bfloat16)
    if c.get("residual"):
        t["r"] = _randn(seed, 8, M, N).to(torch.bfloat16)
    if k in ("rope", "conv"):
        t["pos"] = torch.from_numpy(positions(_lengths(seed, M))).to(DEV)
    return t


def prepare(c, seed):
    k = c["kind"]
    t = _inputs(c, seed)
    if k == "stack":
        from sys1_amd.device import load
        from sys1_amd.stacks import ProjectionStack, modernbert
        s = ProjectionStack(modernbert(c["hidden"], c["inter"], c["layers"], "encoder"), load(0), c["M"],
                            weights=t["w"], norms=True, norm_weights=t["g"], blocked=c["blocked"])
        return {"call": lambda: s.forward(t["x"], c["M"])}
    if k == "linear":
        from sys1_amd.linear import Linear
        m = Linear(t["w"], t.get("b"), blocked=c["blocked"])
        return {"call": lambda: m(t["x"], t.get("r"), c["act"] or False)}
    if k == "gated":
        from sys1_amd.linear import GatedLinear
        m = GatedLinear(t["w"], c["act"], blocked=c["blocked"])
        return {"call": lambda: m(t["x"])}
    if k == "norm":
        from sys1_amd.norm import NormLinear
        eps = 1e-5 if c["norm"] == "layer" else 1e-6
        m = NormLinear(t["w"], t["g"], c["norm"], eps, c["act"] or None, blocked=c["blocked"])
        return {"call": lambda: m(t["x"])}
    if k == "rope":
        from sys1_amd.rope import RopeQkvLinear, rope_tables
        m = RopeQkvLinear(t["w"], c["heads"], *rope_tables(160000.0, 64, 8192, DEV))
        return {"call": lambda: m(t["x"], t["pos"])}
    from sys1_amd.deltanet import InProjConv
    m = InProjConv(t["w"], t["cw"], c["C"], t["g"], 1e-6)
    return {"call": lambda: m(t["x"], t["pos"])}


def run(state):
    return state["call"]()


def _norm64(x, g, kind):
    if kind == "layer":
        x = x - x.mean(1, keepdim=True)
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-5) * g.double()
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-6) * (1.0 + g.double())


def _act64(v, act):
    if act in ("erf", "gelu"):
        return 0.5 * v * (1.0 + torch.erf(v / math.sqrt(2.0)))
    if act == "tanh":
        return 0.5 * v * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (v + 0.044715 * v ** 3)))
    if act == "silu":
        return v * torch.sigmoid(v)
    return v


def _gated64(p, act):
    g, u = p.chunk(2, dim=1)
    return _act64(g, act) * u


def exact(c, seed):
    t = _inputs(c, seed)
    k = c["kind"]
    x = t["x"].double()
    if k == "stack":
        H = c["hidden"]
        for w, g in zip(t["w"], t["g"]):
            wqkv, wo, wi, w2 = (v.double() for v in w)
            a = _norm64(x, g[0], "layer") if g[0] is not None else x
            x = x + (a @ wqkv.T)[:, 2 * H:] @ wo.T
            x = x + _gated64(_norm64(x, g[2], "layer") @ wi.T, "gelu") @ w2.T
        return x
    if k == "norm":
        x = _norm64(x, t["g"], c["norm"])
    if k == "conv" and c["norm"]:
        x = _norm64(x, t["g"], "rms")
    y = x @ t["w"].double().T
    if k in ("gated", "norm") and c["act"]:
        return _gated64(y, c["act"])
    if "b" in t:
        y = y + t["b"].double()
    if k == "linear":
        y = _act64(y, c["act"])
    if "r" in t:
        y = y + t["r"].double()
    if k == "rope":
        M, H = c["M"], 64 * c["heads"]
        inv = 1.0 / torch.pow(torch.tensor(160000.0, dtype=torch.float64), torch.arange(0, 64, 2) / 64.0).float()
        # the f32 frequencies of the reference's tables
        f = (t["pos"].cpu().float()[:, None] * inv[None, :]).double().to(DEV)
        cos, sin = f.cos()[:, None, :], f.sin()[:, None, :]
        q = y.reshape(M, 3, c["heads"], 64).permute(1, 0, 2, 3).clone()
        a, b = q[:2, ..., :32].clone(), q[:2, ..., 32:].clone()
        q[:2, ..., :32], q[:2, ..., 32:] = a * cos - b * sin, a * sin + b * cos
        return q.reshape(3, M, H)
    if k == "conv":
        C, pos = c["C"], t["pos"][:, None]
        p, cw = y[:, :C], t["cw"].double()
        out = p * cw[:, 3]
        for s in range(1, 4):
            if c["M"] > s:
                out[s:] += torch.where(pos[s:] >= s, p[:-s], torch.zeros_like(p[:-s])) * cw[:, 3 - s]
        y[:, :C] = _act64(out, "silu")
    return y
