"""The work this framework is used for, as measurable cases.

Each case goes through the public entry points: the recurrence as an op
(``chunk_kda`` / ``chunk_gdn``, forward or forward + VJP by autograd), the
``GatedDeltaLayer`` around it (inference and training) and the video classifier.
A case is a dict of plain values:

* ``kind``: "kda" (per-channel decay), "gdn" (one decay per head), "layer",
  "model";
* ``B, T, H, D``: sequences, tokens, heads, head size (``model``: B clips; the
  other sizes are the model's);
* ``dtype``: of the activations, "bf16" or "fp32"; ``g``: of the decay;
* ``decay``: "mild" (g = -0.1 softplus(N(0, 1)), the op benchmark's) or "layer"
  (g = -A_h softplus(N(0, 0.5^2)), A_h ~ U[1, 16], the layer's at initialisation);
* ``state``: an initial state is carried in; ``train``: forward and VJP.
"""
import math

import torch
import torch.nn.functional as F
from torch.utils.checkpoint import checkpoint

from mlx_vit_amd import GatedDeltaLayer, chunk_gdn, chunk_kda
from mlx_vit_amd.model import config4, to_bf16

DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
DEVICE = "cuda"
MODEL = dict(layers=12, embed=384, dim=768, heads=12, head_dim=64, tokens=1568, patch=2 * 16 * 16 * 3)


def _op(name, B, T, H, D, dtype="bf16", g="bf16", decay="mild", state=False, train=False, kind="kda"):
    c = dict(kind=kind, B=B, T=T, H=H, D=D, dtype=dtype, g=g, decay=decay, state=state, train=train)
    return dict(name=name, **c) if name else c


def _layer(name, B, T, H, D, dtype="bf16", state=False, train=True):
    return _op(name, B, T, H, D, dtype, "fp32", "layer", state, train, "layer")


def listed():
    return [
        # one short clip of a small model checked in fp32: latency and launches
        _op("op-fwd-small-fp32", 1, 256, 2, 64, "fp32", "fp32"),
        # the op's forward at the ViT-B token shape: 8 tubelets x 14 x 14 patches, 8 clips
        _op("op-fwd-vitb", 8, 1568, 12, 64),
        # the headline: forward + VJP at that shape
        _op("op-train-vitb", 8, 1568, 12, 64, train=True),
        # the default classifier's layer (32 frames, width 384: 6 heads, 3136 tokens), fp32 g as
        # the layer produces it, at the layer's initial decay
        _op("op-train-default-layerdecay", 8, 3136, 6, 64, g="fp32", decay="layer", train=True),
        # training in fp32 (the reference's parity mode), a small batch
        _op("op-train-fp32", 2, 1568, 6, 64, "fp32", "fp32", "layer", train=True),
        # a long stream with its state carried in and out, D = 128
        _op("op-fwd-long-d128", 1, 32768, 16, 128, state=True),
        # the SSv2 model's layer: 8 heads of 96
        _op("op-train-ssv2-d96", 8, 1568, 8, 96, g="fp32", decay="layer", train=True),
        # the scalar-alpha sibling at the ViT-B shape
        _op("op-train-gdn", 8, 1568, 12, 64, g="bf16", train=True, kind="gdn"),
        # one layer of the ViT-B classifier, trained
        _layer("layer-train-vitb", 8, 1568, 12, 64),
        # the same tokens with the time-only scan: one sequence of 8 tubelets per spatial location
        _layer("layer-train-temporal", 8 * 196, 8, 12, 64),
        # streaming inference: the next tubelet's 196 tokens of one clip, the state carried
        _layer("layer-stream", 1, 196, 12, 64, state=True, train=False),
        # classifying a batch of clips with the 12-layer model
        dict(name="model-classify", kind="model", B=8, dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["kda", "kda", "kda", "kda", "gdn", "layer", "layer", "temporal", "stream", "model"])
    if kind == "model":
        return dict(kind="model", B=rng.randint(1, 7), dtype="bf16")
    if kind in ("layer", "stream", "temporal"):
        D = rng.choice([64, 64, 64, 96, 32])
        H = rng.randint(3, 768 // D)
        if kind == "stream":
            return _layer(None, rng.randint(1, 2), _log_int(rng, 1, 400), H, D, "bf16", True, False)
        if kind == "temporal":
            return _layer(None, rng.randint(1, 8) * 196, rng.randint(4, 8), H, D)
        return _layer(None, rng.randint(1, 8), _log_int(rng, 100, 1568), H, D, rng.choice(["bf16", "bf16", "bf16", "fp32"]))
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
    train = rng.random() < 0.6
    if kind == "gdn":
        D, H = rng.choice([32, 64, 64]), rng.randint(2, 12)
        return _op(None, rng.randint(1, 8), _log_int(rng, 50, 1568), H, D, dtype, "bf16", "mild", False, train, "gdn")
    D = rng.choice([32, 64, 64, 64, 96, 128])
    H = rng.randint(1, 12 * 64 // max(D, 64))
    g = "fp32" if dtype == "fp32" else rng.choice(["bf16", "fp32"])
    B = 1 if rng.random() < 0.3 else rng.randint(2, 8)
    T = _log_int(rng, 64, 8192 if B == 1 else 1568)
    return _op(None, B, T, H, D, dtype, g, rng.choice(["mild", "layer"]), rng.random() < 0.3, train)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device=DEVICE)


def _op_inputs(case, seed):
    """The op's operands by name, None where the case has none."""
    B, T, H, D = (case[n] for n in "BTHD")
    dt, gen = DTYPES[case["dtype"]], _gen(seed)
    x = {}
    x["q"] = F.normalize(_randn(gen, B, T, H, D), dim=-1).to(dt)
    x["k"] = F.normalize(_randn(gen, B, T, H, D), dim=-1).to(dt)
    x["v"] = _randn(gen, B, T, H, D).to(dt)
    if case["kind"] == "gdn":
        x["g"] = torch.sigmoid(0.6 * _randn(gen, B, T, H)).to(dt)       # alpha = sigmoid(a_proj(x))
    elif case["decay"] == "mild":
        x["g"] = (-0.1 * F.softplus(_randn(gen, B, T, H, D))).to(DTYPES[case["g"]])
    else:
        A = 1 + 15 * torch.rand(H, 1, generator=gen, device=DEVICE)
        x["g"] = (-A * F.softplus(0.5 * _randn(gen, B, T, H, D))).to(DTYPES[case["g"]])
    x["beta"] = torch.sigmoid(_randn(gen, B, T, H)).to(dt)
    x["s0"] = 0.02 * _randn(gen, B, H, D, D) if case["state"] else None
    x["do"] = _randn(gen, B, T, H, D).to(dt) if case["train"] else None
    return x


def _module(build, seed, dtype):
    """A module with the reference's initialisation, drawn from the seed."""
    with torch.random.fork_rng(devices=[]):
        torch.manual_seed(seed)
        m = build()
    return (to_bf16(m) if dtype == "bf16" else m).to(DEVICE)


def _make_layer(case, seed):
    return _module(lambda: GatedDeltaLayer(case["H"] * case["D"], case["H"], case["D"]), seed, case["dtype"])


def _layer_inputs(case, seed):
    B, T, H, D = (case[n] for n in "BTHD")
    dt, gen = DTYPES[case["dtype"]], _gen(seed)
    x = _randn(gen, B, T, H * D).to(dt)                                  # the block's LayerNorm output
    s0 = 0.02 * _randn(gen, B, H, D, D) if case["state"] else None
    dout = _randn(gen, B, T, H * D).to(dt) if case["train"] else None
    return x, s0, dout


def _clips(case, seed):
    return _randn(_gen(seed), case["B"], 16, 224, 224, 3).to(DTYPES[case["dtype"]])


def prepare(case, seed):
    if case["kind"] == "model":
        return dict(case=case, model=_module(config4, seed, case["dtype"]).eval(), video=_clips(case, seed))
    if case["kind"] == "layer":
        x, s0, dout = _layer_inputs(case, seed)
        layer = _make_layer(case, seed)
        return dict(case=case, layer=layer, x=x.requires_grad_(case["train"]), s0=s0, dout=dout,
                    params=list(layer.parameters()))
    x = _op_inputs(case, seed)
    leaves = [x[n] for n in ("q", "k", "v", "g", "beta", "s0") if x[n] is not None]
    if case["train"]:
        for t in leaves:
            t.requires_grad_(True)
    return dict(case=case, x=x, leaves=leaves)


def run(state):
    case = state["case"]
    if case["kind"] == "model":
        with torch.no_grad():
            return state["model"](state["video"])
    if case["kind"] == "layer":
        if not case["train"]:
            with torch.no_grad():
                return state["layer"](state["x"], state["s0"])
        out, s = state["layer"](state["x"])
        return [out, s, *torch.autograd.grad(out, [state["x"], *state["params"]], state["dout"])]
    x = state["x"]
    op = chunk_gdn if case["kind"] == "gdn" else chunk_kda
    o, s = op(x["q"], x["k"], x["v"], x["g"], x["beta"], x["s0"])
    if not case["train"]:
        return [o, s]
    return [o, s, *torch.autograd.grad(o, state["leaves"], x["do"])]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _recurrence_flops(n, T, D, train):
    """n token-heads of the chunkwise form, chunks of min(T, 64): 10 C D + 6 D^2 +
    (2/3) C^2 forward, twice that backward."""
    C = min(T, 64)
    return n * (10 * C * D + 6 * D * D + 2 / 3 * C * C) * (3 if train else 1)


def work(case):
    es = 2 if case["dtype"] == "bf16" else 4
    if case["kind"] == "model":
        m, n = MODEL, case["B"] * MODEL["tokens"]
        weights = m["embed"] * (m["patch"] + m["dim"]) + m["layers"] * (12 * m["dim"] ** 2 + 4 * m["head_dim"] * m["dim"])
        video = case["B"] * 16 * 224 * 224 * 3
        return {"bytes": es * (weights + video),
                "flops": 2 * n * weights + m["layers"] * _recurrence_flops(n * m["heads"], m["tokens"], m["head_dim"], False)}
    B, T, H, D, train = case["B"], case["T"], case["H"], case["D"], case["train"]
    n, states = B * T * H, B * H * D * D * 4
    if case["kind"] == "layer":
        w, tok = 4 * (H * D) ** 2 + 4 * D * H * D + 17 * H * D, n * D
        flops = 2 * B * T * w * (3 if train else 1) + _recurrence_flops(n, T, D, train)
        state_bytes = states * (2 if case["state"] else 1)
        if not train:
            return {"bytes": es * (w + 2 * tok) + state_bytes, "flops": flops}
        return {"bytes": es * (2 * w + 4 * tok) + state_bytes, "flops": flops}
    gb = n * es if case["kind"] == "gdn" else n * D * (2 if case["g"] == "bf16" else 4)
    ins = n * (3 * D + 1) * es + gb + (states if case["state"] else 0)
    outs = n * D * es + states
    if train:
        outs += ins                                                      # a gradient for every input
        ins += n * D * es                                                # do
    return {"bytes": ins + outs, "flops": _recurrence_flops(n, T, D, train)}


# ---------------------------------------------------------------------------
# the same results in 64 bits, by plain torch: the recurrence token by token
# ---------------------------------------------------------------------------
def _steps(S, q, k, v, eg, beta):
    """Tokens of the rows q, k, v, eg (T, N, D), beta (T, N): S <- S diag(e^g);
    S <- S (I - beta k k^T) + beta v k^T; o = S q, S (N, D, D) with S[v][k]."""
    out = []
    for t in range(q.shape[0]):
        S = S * eg[t].unsqueeze(-2)
        u = beta[t].unsqueeze(-1) * (v[t] - (S * k[t].unsqueeze(-2)).sum(-1))
        S = S + u.unsqueeze(-1) * k[t].unsqueeze(-2)
        out.append((S * q[t].unsqueeze(-2)).sum(-1))
    return torch.stack(out), S


def _recurrence64(q, k, v, g, beta, s0):
    """(B, T, H, D) fp64 operands -> o (B, T, H, D), final state (B, H, D, D)."""
    B, T, H, D = q.shape
    rows = [t.transpose(0, 1).reshape(T, B * H, -1) for t in (q, k, v, torch.exp(g))]
    bt = beta.transpose(0, 1).reshape(T, B * H)
    S = torch.zeros(B * H, D, D, dtype=q.dtype, device=q.device) if s0 is None else s0.reshape(B * H, D, D)
    outs = []
    for a in range(0, T, 64):
        part = [t[a:a + 64] for t in rows] + [bt[a:a + 64]]
        o, S = checkpoint(_steps, S, *part, use_reentrant=False) if torch.is_grad_enabled() else _steps(S, *part)
        outs.append(o)
    o = torch.cat(outs).reshape(T, B, H, D).transpose(0, 1)
    return o, S.reshape(B, H, D, D)


def _layer64(p, x, H, D, s0):
    """GatedDeltaLayer.forward on fp64 parameters p (by name)."""
    B, T, HD = x.shape

    def conv(n):
        y = F.pad(x @ p[n + "_proj.weight"].T, (0, 0, 3, 0))
        w = p[n + "_conv1d.weight"].reshape(HD, 4)
        return F.silu(sum(y[:, i:i + T] * w[:, i] for i in range(4)) + p[n + "_conv1d.bias"])

    q, k, v = conv("q"), conv("k"), conv("v")
    q, k = F.normalize(q, dim=-1) * D ** -0.5, F.normalize(k, dim=-1)
    f = (x @ p["f_proj_1.weight"].T) @ p["f_proj_2.weight"].T + p["dt_bias"]
    g = -torch.exp(p["A_log"]).reshape(H, 1) * F.softplus(f.reshape(B, T, H, D))
    beta = torch.sigmoid(x @ p["b_proj.weight"].T)
    o, s = _recurrence64(*(t.reshape(B, T, H, D) for t in (q, k, v)), g, beta, s0)
    gate = (x @ p["g_proj_1.weight"].T) @ p["g_proj_2.weight"].T + p["g_proj_2.bias"]
    y = o * torch.rsqrt(o.square().mean(-1, keepdim=True) + 1e-5) * p["o_norm.weight"]
    return (y.reshape(B, T, HD) * torch.sigmoid(gate)) @ p["o_proj.weight"].T, s


def _model64(p, video, heads, head_dim):
    B, Tf, Hh, Ww, C = video.shape
    x = video.reshape(B, Tf // 2, 2, Hh // 16, 16, Ww // 16, 16, C).permute(0, 1, 3, 5, 2, 4, 6, 7)
    w = p["backbone.encoder.tubelet_embed.projection.weight"]
    x = x.reshape(B, -1, 2 * 16 * 16 * C) @ w.reshape(w.shape[0], -1).T + p["backbone.encoder.tubelet_embed.projection.bias"]

    def norm(t, n):
        return F.layer_norm(t, t.shape[-1:], p[n + ".weight"], p[n + ".bias"], 1e-6)

    x = norm(x, "backbone.encoder.norm") @ p["backbone.dim_proj.weight"].T + p["backbone.dim_proj.bias"]
    for i in range(MODEL["layers"]):
        b = "backbone.processor_blocks.%d." % i
        lp = {n[len(b) + 6:]: t for n, t in p.items() if n.startswith(b + "layer.")}
        x = x + _layer64(lp, norm(x, b + "norm1"), heads, head_dim, None)[0]
        h = F.gelu(norm(x, b + "norm2") @ p[b + "mlp.0.weight"].T + p[b + "mlp.0.bias"])
        x = x + h @ p[b + "mlp.3.weight"].T + p[b + "mlp.3.bias"]
    x = norm(x, "backbone.processor_norm")
    D = x.shape[-1]
    frames = x.reshape(B, Tf // 2, -1, D).mean(2)
    q = p["head.temporal_query"].reshape(1, heads, 1, -1)
    k, v = ((frames @ p["head.t_proj_%s.weight" % n].T).reshape(B, Tf // 2, heads, -1).transpose(1, 2) for n in "kv")
    a = torch.softmax((q * k).sum(-1) * (D // heads) ** -0.5, -1)
    out = (a.unsqueeze(-1) * v).sum(2).reshape(B, D) @ p["head.t_proj_out.weight"].T + frames.mean(1)
    return norm(out, "head.t_norm") @ p["head.fc.weight"].T + p["head.fc.bias"]


def exact(case, seed):
    if case["kind"] == "model":
        p = {n: t.detach().double() for n, t in _module(config4, seed, case["dtype"]).named_parameters()}
        with torch.no_grad():
            return _model64(p, _clips(case, seed).double(), MODEL["heads"], MODEL["head_dim"])
    train = case["train"]
    with torch.set_grad_enabled(train):
        if case["kind"] == "layer":
            x, s0, dout = _layer_inputs(case, seed)
            p = {n: t.detach().double().requires_grad_(train) for n, t in _make_layer(case, seed).named_parameters()}
            x = x.double().requires_grad_(train)
            out, s = _layer64(p, x, case["H"], case["D"], None if s0 is None else s0.double())
            if not train:
                return [out, s]
            return [out.detach(), s.detach(), *torch.autograd.grad(out, [x, *p.values()], dout.double())]
        t = {n: None if v is None else v.double() for n, v in _op_inputs(case, seed).items()}
        leaves = [t[n].requires_grad_(train) for n in ("q", "k", "v", "g", "beta", "s0") if t[n] is not None]
        g = t["g"]
        if case["kind"] == "gdn":
            g = torch.log(g).unsqueeze(-1).expand(t["q"].shape)
        o, s = _recurrence64(t["q"], t["k"], t["v"], g, t["beta"], t["s0"])
        if not train:
            return [o, s]
        return [o.detach(), s.detach(), *torch.autograd.grad(o, leaves, t["do"])]


def tolerance(case):
    """About four times the largest error against ``exact`` over the outputs: fp32
    operands (split-bf16 products) 7e-6; bf16 operands with fp32 sums 4.3e-3 for
    the op, 7e-3 for a layer between its GEMMs and for the model's logits."""
    if case["dtype"] == "fp32":
        return {"rel": 3e-5}
    return {"rel": 1.8e-2 if case["kind"] in ("kda", "gdn") else 2.8e-2}
