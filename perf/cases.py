"""What users of this package run, as timed cases: the SVDQuant linear (W4A4 and W4A16) at the
layer shapes of a Krea-2 block from a handful of prompt tokens to a 2048-pixel latent, the sibling
launches, the block's attention and its normalizations, and a whole block.

``listed()`` names the cases, ``draw(rng)`` gives further ones of the same ranges, ``prepare`` /
``run`` make one and take it through the public entry points, ``exact`` evaluates it in 64 bits
with plain torch.  All sizes are the package's own: the layer shapes of ``Krea2Dims``, group 64 and
128 (the benchmark's and the quantizer's default), ranks 32 and 64 (the attention and MLP
defaults), LoRA rank 64 (the benchmark's), 2304 / 4096 / 16384 latent tokens (768, 1024 and 2048
pixels) with prompt tokens beside them.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from krea2_svdquant_amd import SVDQuantLinear
from krea2_svdquant_amd.runtime import krea2_standin as standin
from krea2_svdquant_amd.runtime.siblings import run_grouped

HIDDEN, HEADS, KV_HEADS, HEAD_DIM, MLP = 6144, 48, 12, 128, 16384
KV = KV_HEADS * HEAD_DIM
# (out_features, in_features) of the quantized linears of a block
SHAPES = {"to_q": (HIDDEN, HIDDEN), "to_k": (KV, HIDDEN), "to_out": (HIDDEN, HIDDEN), "ff.up": (MLP, HIDDEN),
          "ff.down": (HIDDEN, MLP)}
ATTN_INPUTS, FF_INPUTS = (HIDDEN, HIDDEN, KV, KV), (MLP, MLP)   # to_q, to_gate, to_k, to_v; ff.up, ff.gate
BACKENDS = {"w4a4": "hip_gfx950", "w4a16": "hip_gfx950_w4a16"}


def _linear(name, mode, m, layer, group, rank, lora=0, bias=False):
    n, k = SHAPES[layer]
    return {"name": name, "kind": "linear", "mode": mode, "m": m, "n": n, "k": k, "group": group, "rank": rank,
            "lora": lora, "bias": bias}


def listed():
    return [
        # the key projection of a short prompt: the smallest call of a block, latency and launches
        _linear("prompt to_k", "w4a4", 64, "to_k", 64, 32),
        # a 256-token prompt through a square projection (the benchmark's smallest configuration)
        _linear("prompt to_q", "w4a4", 256, "to_q", 64, 32),
        # a 77-token prompt through the MLP of a bf16-activation layer, quantizer defaults (group
        # 128, MLP rank 64)
        _linear("prompt ff.up w4a16", "w4a16", 77, "ff.up", 128, 64),
        # the headline layer: ff.up over the 4096 latent tokens of a 1024-pixel image
        _linear("image ff.up", "w4a4", 4096, "ff.up", 64, 32),
        # 768-pixel image with a 77-token prompt: a row count that no tile divides, quantizer
        # defaults, the long reduction
        _linear("ragged ff.down", "w4a4", 2381, "ff.down", 128, 64),
        # the bf16-activation benchmark: ff.up over a 768-pixel image's latent tokens
        _linear("image ff.up w4a16", "w4a16", 2304, "ff.up", 64, 32),
        # a 2048-pixel image with a LoRA adapter fused into ff.down: the largest call
        _linear("lora ff.down", "w4a4", 16384, "ff.down", 64, 32, lora=64),
        # to_q, to_gate, to_k and to_v of one block over latent and prompt tokens, grouped
        {"name": "attention inputs", "kind": "siblings", "mode": "w4a4", "set": "attn", "m": 4352, "group": 64,
         "rank": 32},
        # the block's attention over a 1024-pixel image with its prompt
        {"name": "attention", "kind": "attention", "t": 4352},
        # the same for a 512-pixel image and a 77-token prompt: short and ragged
        {"name": "ragged attention", "kind": "attention", "t": 1101},
        # the gated residual and adaptive norm between two blocks: a pass over memory
        {"name": "residual norm", "kind": "norm", "t": 4352},
        # one whole denoiser block with bf16 activations over a 768-pixel image and a 77-token prompt
        {"name": "block w4a16", "kind": "block", "mode": "w4a16", "t": 2381, "group": 64, "rank": 32},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same kinds: token counts log-uniform (odd ones among them, one in four a multiple
    of 64), the block's layers or, one in five, another width."""
    kind = rng.choice(["linear"] * 6 + ["siblings", "siblings", "attention", "norm", "block"])

    def tokens(lo, hi):
        m = _log_int(rng, lo, hi)
        return max(64, m // 64 * 64) if m >= 64 and rng.random() < 0.25 else m

    if kind == "linear":
        n, k = SHAPES[rng.choice(sorted(SHAPES))]
        if rng.random() < 0.2:
            n, k = _log_int(rng, 256, 8192), 64 * _log_int(rng, 8, 128)
        return {"kind": kind, "mode": rng.choice(["w4a4", "w4a4", "w4a16"]), "m": tokens(16, 12288), "n": n, "k": k,
                "group": rng.choice([64, 128]), "rank": rng.choice([32, 64]),
                "lora": rng.choice([0, 0, 0, 16, 64]), "bias": rng.random() < 0.3}
    if kind == "siblings":
        return {"kind": kind, "mode": rng.choice(["w4a4", "w4a4", "w4a16"]), "set": rng.choice(["attn", "ff"]),
                "m": tokens(32, 4608), "group": rng.choice([64, 128]), "rank": rng.choice([32, 64])}
    if kind == "attention":
        return {"kind": kind, "t": tokens(64, 8192)}
    if kind == "norm":
        return {"kind": kind, "t": tokens(64, 16384)}
    return {"kind": kind, "mode": "w4a16", "t": tokens(128, 4608), "group": rng.choice([64, 128]), "rank": 32}


# ---- inputs ------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g)


def _activation(g, m, k):
    """bf16 activations as a transformer's linears meet them: N(0, 1) with 1% outlier channels."""
    x = _randn(g, m, k)
    hot = torch.randperm(k, device="cuda", generator=g)[: max(1, k // 100)]
    x[:, hot] *= 12.0
    return x.to(torch.bfloat16)


def _layer(g, n, k, case):
    state = standin.random_quantized_state(n, k, rank=case["rank"], group_size=case["group"], device="cuda",
                                           generator=g)
    if case.get("bias"):
        state.bias = _randn(g, n).to(torch.bfloat16)
    layer = SVDQuantLinear(state, backend=BACKENDS[case["mode"]])
    if case.get("lora"):
        r = case["lora"]
        layer.add_lora_adapter((_randn(g, r, k) * 0.01).to(torch.bfloat16), (_randn(g, n, r) * 0.01).to(torch.bfloat16),
                               scale=0.8)
    return layer


def _inputs(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "linear":
        return {"layers": [_layer(g, case["n"], case["k"], case)], "x": _activation(g, case["m"], case["k"])}
    if kind == "siblings":
        ns = ATTN_INPUTS if case["set"] == "attn" else FF_INPUTS
        return {"layers": [_layer(g, n, HIDDEN, case) for n in ns], "x": _activation(g, case["m"], HIDDEN)}
    if kind == "attention":   # q and k as the per-head norm leaves them, v as a projection does
        t = case["t"]
        q, k, v = _randn(g, t, HEADS, HEAD_DIM), _randn(g, t, KV_HEADS, HEAD_DIM), _randn(g, t, KV_HEADS, HEAD_DIM)
        return {"q": F.rms_norm(q, (HEAD_DIM,)).to(torch.bfloat16), "k": F.rms_norm(k, (HEAD_DIM,)).to(torch.bfloat16),
                "v": v.to(torch.bfloat16)}
    if kind == "norm":
        t = case["t"]
        vec = {name: (_randn(g, HIDDEN) * 0.1).to(torch.bfloat16) for name in ("gate", "scale", "shift")}
        return {"x": _activation(g, t, HIDDEN), "y": _randn(g, t, HIDDEN).to(torch.bfloat16), **vec,
                "weight": 1 + vec["scale"]}
    dims = standin.Krea2Dims(layers=1)
    model = standin.Krea2StandInTransformer.random(dims, rank=case["rank"], group_size=case["group"],
                                                   backend=BACKENDS[case["mode"]], device="cuda", seed=int(seed))
    return {"model": model, "x": _randn(g, case["t"], HIDDEN).to(torch.bfloat16)}


def prepare(case, seed):
    """Inputs, and layers that have answered a call before (a layer builds its kernel operands on
    its first call and keeps them)."""
    state = dict(_inputs(case, seed), case=case)
    if case["kind"] in ("linear", "siblings", "block"):
        with torch.no_grad():
            run(state)
    return state


@torch.no_grad()
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        return state["layers"][0](state["x"])
    if kind == "siblings":
        return run_grouped(state["x"], state["layers"])
    if kind == "attention":
        return standin.attention(state["q"], state["k"], state["v"])
    if kind == "norm":
        return list(standin.residual_norm_modulate(state["x"], state["gate"], state["y"], state["scale"],
                                                   state["shift"], weight=state["weight"]))
    return state["model"](state["x"])


# ---- what a pass cannot do without -----------------------------------------------------------
def _linear_work(m, n, k, group, rank, lora):
    r = rank + lora
    weights = n * k // 2 + 2 * n * (k // group) + 2 * r * (n + k) + 2 * k
    return {"bytes": 2 * m * k + weights + 2 * m * n, "flops": 2 * m * n * k + 2 * m * r * (n + k)}


def work(case):
    kind = case["kind"]
    if kind == "linear":
        return _linear_work(case["m"], case["n"], case["k"], case["group"], case["rank"], case["lora"])
    if kind == "siblings":
        ns = ATTN_INPUTS if case["set"] == "attn" else FF_INPUTS
        parts = [_linear_work(case["m"], n, HIDDEN, case["group"], case["rank"], 0) for n in ns]
        shared = (len(ns) - 1) * 2 * case["m"] * HIDDEN          # the layers read one x
        return {"bytes": sum(p["bytes"] for p in parts) - shared, "flops": sum(p["flops"] for p in parts)}
    t = case["t"]
    if kind == "attention":
        return {"bytes": 2 * t * HEAD_DIM * (2 * HEADS + 2 * KV_HEADS), "flops": 4 * t * t * HEAD_DIM * HEADS}
    if kind == "norm":
        return {"bytes": 4 * 2 * t * HIDDEN + 3 * 2 * HIDDEN, "flops": 8 * t * HIDDEN}
    shapes = [(HIDDEN, HIDDEN)] * 3 + [(KV, HIDDEN)] * 2 + [(MLP, HIDDEN)] * 2 + [(HIDDEN, MLP)]
    parts = [_linear_work(t, n, k, case["group"], case["rank"], 0) for n, k in shapes]
    weights = sum(p["bytes"] for p in parts) - sum(2 * t * (n + k) for n, k in shapes)
    return {"bytes": weights + 2 * 2 * t * HIDDEN,
            "flops": sum(p["flops"] for p in parts) + 4 * t * t * HEAD_DIM * HEADS}


def tolerance(case):
    """About four times what the path measures against ``exact``.  Linears: one bf16 rounding of the
    output (2-norm 1.7e-3, at most half a unit in the last place, 3.9e-3 of a value).  The norm's
    second output rounds twice (2.4e-3, 7.7e-3), the attention rounds its probabilities as well
    (2.3e-3, 1.1e-2).  A block chains a dozen of these (6.2e-3, 3.7e-2)."""
    rel, most = {"linear": (7e-3, 1.6e-2), "siblings": (7e-3, 1.6e-2), "attention": (1e-2, 4.5e-2),
                 "norm": (1e-2, 3e-2), "block": (2.4e-2, 0.15)}[case["kind"]]
    return {"rel": rel, "max": most}


# ---- the same in 64 bits -----------------------------------------------------------------------
def _unpack(qweight):
    """Packed codes [N, K/2] -> float64 [N, K]: byte j holds q[2j] + 8 in its low nibble."""
    lo, hi = qweight & 15, qweight >> 4
    return torch.stack((lo, hi), -1).reshape(qweight.shape[0], -1).double() - 8.0


def _linear_exact(x, layer):
    """The layer's output in 64 bits: x / s rounded to bf16, codes of the dynamic per-group
    quantizer (bf16 scales, nearest even), everything after that in float64."""
    s = layer.state
    g, k = s.group_size, s.original_shape[1]
    kp = s.qweight.shape[1] * 2
    x_hat = F.pad((x.float() / s.smooth_scale.float()).to(torch.bfloat16), (0, kp - k))
    codes = _unpack(s.qweight).view(-1, kp // g, g)
    if layer.backend.value == BACKENDS["w4a16"]:
        sw = s.weight_scales.to(torch.bfloat16).float().unsqueeze(-1)
        w = (codes.float() * sw).to(torch.bfloat16).double().reshape(-1, kp)
        a = x_hat.double()
    else:
        grp = x_hat.view(x.shape[0], kp // g, g)
        eps = torch.tensor(1e-8, dtype=torch.bfloat16, device=x.device)
        sx = (torch.maximum(grp.abs().amax(-1, keepdim=True), eps).float() / 7.0).to(torch.bfloat16)
        q = torch.round(grp.float() / sx.float()).clamp_(-8, 7)
        a = (q.double() * sx.double()).reshape(x.shape[0], kp)
        w = (codes * s.weight_scales.double().unsqueeze(-1)).reshape(-1, kp)
    y = a @ w.t()
    del a, w, codes
    y += (x_hat[:, :k].double() @ s.l2.double().t()) @ s.l1.double().t()
    for ad in layer.lora_adapters:
        y += ((x.double() @ ad.down_weight.double().t()) @ ad.up_weight.double().t()) * ad.multiplier
    if s.bias is not None:
        y += s.bias.double()
    return y


def _attention_exact(q, k, v):
    t, heads = q.shape[0], q.shape[1]
    out = torch.empty(t, heads, HEAD_DIM, dtype=torch.float64, device=q.device)
    for h in range(heads):
        kh, vh = (z[:, h // (heads // k.shape[1])].double() for z in (k, v))
        p = torch.softmax(q[:, h].double() @ kh.t() / math.sqrt(HEAD_DIM), -1)
        out[:, h] = p @ vh
    return out.reshape(t, heads * HEAD_DIM)


def _norm_exact(x, weight, shift, eps=1e-6):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * weight.double() + shift.double()


def _rope_exact(t, eps=1e-6):
    """Per-head RMS norm and the rotate-half rotary embedding of bf16 [T, heads, d]."""
    t = t.double()
    t = (t * torch.rsqrt(t.square().mean(-1, keepdim=True) + eps)).to(torch.bfloat16).double()
    cos, sin = standin.rope_tables(t.shape[0], HEAD_DIM, t.device, torch.bfloat16)
    h = HEAD_DIM // 2
    c, s = cos[:, None, :h].double(), sin[:, None, :h].double()
    t1, t2 = t[..., :h], t[..., h:]
    return torch.cat((t1 * c - t2 * s, t2 * c + t1 * s), -1)


def _block_exact(x, block):
    """One block without its last rounding, each op in 64 bits on the bf16 values that the op before it hands over."""
    bf = torch.bfloat16
    lin = block.linears()
    shift_a, scale_a, gate_a, shift_f, scale_f, gate_f = block.modulation
    t = x.shape[0]

    def apply(name, z):
        return _linear_exact(z, lin[name]).to(bf)

    h = _norm_exact(x, 1 + scale_a, shift_a).to(bf)
    q, k, v = (apply("attn." + n, h).view(t, -1, HEAD_DIM) for n in ("to_q", "to_k", "to_v"))
    a = _attention_exact(_rope_exact(q).to(bf), _rope_exact(k).to(bf), v).to(bf)
    a = (a.double() * torch.sigmoid(apply("attn.to_gate", h).double()).to(bf).double()).to(bf)
    x = (x.double() + gate_a.double() * apply("attn.to_out.0", a).double()).to(bf)
    h = _norm_exact(x, 1 + scale_f, shift_f).to(bf)
    f = (F.silu(apply("ff.gate", h).double()).to(bf).double() * apply("ff.up", h).double()).to(bf)
    return x.double() + gate_f.double() * apply("ff.down", f).double()


@torch.no_grad()
def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "linear":
        return _linear_exact(s["x"], s["layers"][0])
    if kind == "siblings":
        return [_linear_exact(s["x"], layer) for layer in s["layers"]]
    if kind == "attention":
        return _attention_exact(s["q"], s["k"], s["v"])
    if kind == "norm":
        xo = s["x"].double() + s["gate"].double() * s["y"].double()
        return [xo, _norm_exact(xo.to(torch.bfloat16), s["weight"], s["shift"])]
    return _block_exact(s["x"], s["model"].transformer_blocks[0])
