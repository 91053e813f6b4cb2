"""
Workloads by which the speed of the wide forward is followed.

Every case is one forward of N models through the public entry points (`compile`, the Wide*
modules' `from_modules`, `WideSeqModel`), on inputs resident on the GPU.  `listed()` holds the
fixed cases, `draw(rng)` samples the ranges they stand for, `exact` is the same forward in
64-bit torch.

Families and their declared ranges (sizes spread over their logarithm, odd ones among them):

  mlp        a traced Linear-ReLU-Linear model on the channel-packed input: 4-128 models, batch
             1-256, widths 16-512, fp32 or bf16
  linear     WideLinear over [N, B, F] or [N, B, T, F]: 1-64 models, 1-4096 rows, widths
             16-2048, fp32, bf16 or fp16
  layernorm  WideLayerNorm over [N, B, T, D]: rows of 32-2048 values, fp32 or bf16
  conv       WideConv2d and WideConv1d: 1-128 channels, kernels 1-7, stride 1-2, images of
             7-64 pixels a side (rows of 16-512 in 1-d), fp32, bf16 or fp16
  resblock   a traced conv-BN-ReLU-conv-BN-add-ReLU block on the channel-packed input: 4-100
             models, 16-128 channels, images of 8-56 pixels a side, bf16 or fp32
  attention  WideAttention self-attention: 1-32 models, 1-2048 tokens, head dims 16-128, full
             or causal, fp32, bf16 or fp16
  gru, lstm  WideGRU / WideLSTM: 2-64 models, batch 1-32, 8-128 steps, inputs 16-256 wide,
             hidden sizes 32-512, fp32, bf16 or fp16
  seq        WideSeqModel (embedding, layer norm, LSTM, vocabulary projection), bf16: 2-64
             models, batch 1-16, 8-128 steps, vocabularies 64-8192, hidden 128-512
"""

import math
import os
import sys

import torch
import torch.nn as nn

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "pytorch-parallel-compiler_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DEV = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def listed():
    return [
        # a hundred small ensemble members on one packed batch: one short launch, so dispatch counts
        dict(name="mlp_f32", kind="mlp", dtype="f32", n=100, b=32, i=64, h=128, o=64),
        # the widening layer of a token-wise feed-forward block in fp32, the default dtype
        dict(name="linear_f32", kind="linear", dtype="f32", n=16, b=16, t=128, i=256, o=1024, bias=True),
        # a classifier over 300-wide features and 1000 classes: rows that are no multiple of 16 bytes
        dict(name="linear_ragged_bf16", kind="linear", dtype="bf16", n=20, b=8, t=100, i=300, o=1000, bias=True),
        # the norm between blocks of token models: pure memory traffic
        dict(name="layernorm_f32", kind="layernorm", dtype="f32", n=32, b=8, t=128, d=256),
        # one 3x3 convolution layer of small image models in fp32
        dict(name="conv2d_f32", kind="conv", dtype="f32", n=16, b=8, ci=64, co=64, hh=32, ww=32, kh=3, kw=3,
             stride=1, pad=1),
        # the residual block of a hundred image models in bf16, traced, packed input
        dict(name="resblock_bf16", kind="resblock", dtype="bf16", n=100, b=8, c=64, hw=32),
        # short-sequence self-attention in fp32
        dict(name="attention_f32", kind="attention", dtype="f32", n=32, b=8, s=128, d=256, heads=8, causal=False),
        # encoder self-attention in bf16 at 512 tokens
        dict(name="attention_bf16", kind="attention", dtype="bf16", n=16, b=8, s=512, d=256, heads=8, causal=False),
        # decoder prefill: causal self-attention over 2048 tokens with 64-wide heads
        dict(name="attention_causal_bf16", kind="attention", dtype="bf16", n=4, b=2, s=2048, d=512, heads=8,
             causal=True),
        # a small recurrent model over a short window: a serial chain of 32 steps
        dict(name="gru_f32", kind="gru", dtype="f32", n=32, b=4, t=32, i=64, h=128),
        # a recurrent model whose weights fill more than one compute unit, in fp32
        dict(name="lstm_f32", kind="lstm", dtype="f32", n=16, b=16, t=64, i=128, h=256),
        # whole token models, ids to logits: gather, norm, 128 recurrent steps, vocabulary projection
        dict(name="seq_bf16", kind="seq", dtype="bf16", n=64, b=16, t=128, v=8192, d=256, h=512),
    ]


# ---------------------------------------------------------------------------------------
# drawn cases
# ---------------------------------------------------------------------------------------

def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    """A layer width: mostly a multiple of 16 as configurations have it, now and then any number."""
    w = _log(rng, lo, hi)
    return w if rng.random() < 0.25 else max(lo, min(hi, (w + 8) // 16 * 16))


_LIMITS = {"f32": (1.2e10, 4e9), "bf16": (2.5e11, 4e9), "f16": (2.5e11, 4e9)}   # flops, bytes


def _draw_one(rng):
    kind = rng.choice(["mlp", "linear", "linear", "layernorm", "conv", "conv", "resblock", "attention", "attention",
                       "gru", "lstm", "seq"])
    if kind == "mlp":
        return dict(kind=kind, dtype=rng.choice(["f32", "f32", "bf16"]), n=_log(rng, 4, 128), b=_log(rng, 1, 256),
                    i=_width(rng, 16, 512), h=_width(rng, 16, 512), o=_width(rng, 16, 512))
    if kind == "linear":
        c = dict(kind=kind, dtype=rng.choice(["f32", "f32", "bf16", "bf16", "f16"]), n=_log(rng, 1, 64),
                 b=_log(rng, 1, 64), t=rng.choice([0, _log(rng, 2, 256)]), i=_width(rng, 16, 2048),
                 o=_width(rng, 16, 2048), bias=rng.random() < 0.8)
        return c if c["b"] * max(c["t"], 1) <= 4096 else None
    if kind == "layernorm":
        return dict(kind=kind, dtype=rng.choice(["f32", "bf16"]), n=_log(rng, 1, 64), b=_log(rng, 1, 32),
                    t=_log(rng, 1, 256), d=_width(rng, 32, 2048))
    if kind == "conv":
        k = rng.choice([1, 3, 3, 3, 5, 7])
        c = dict(kind=kind, dtype=rng.choice(["f32", "f32", "bf16", "bf16", "f16"]), n=_log(rng, 1, 32),
                 b=_log(rng, 1, 16), ci=rng.choice([1, 3, 16, 32, 48, 64, 96, 128]),
                 co=rng.choice([16, 32, 40, 64, 96, 128]), kh=k, kw=k, stride=rng.choice([1, 1, 1, 2]), pad=k // 2)
        if rng.random() < 0.3:
            c.update(hh=0, ww=_log(rng, 16, 512), kh=1)              # 1-d
        else:
            c.update(hh=_log(rng, 7, 64), ww=_log(rng, 7, 64))
        return c
    if kind == "resblock":
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "f32"]), n=_log(rng, 4, 100), b=_log(rng, 1, 16),
                    c=rng.choice([16, 32, 48, 64, 64, 96, 128]), hw=_log(rng, 8, 56))
    if kind == "attention":
        heads = rng.choice([1, 2, 4, 8])
        return dict(kind=kind, dtype=rng.choice(["f32", "bf16", "bf16", "f16"]), n=_log(rng, 1, 32), b=_log(rng, 1, 8),
                    s=_log(rng, 1, 2048), d=heads * rng.choice([16, 32, 32, 48, 64, 64, 80, 128]), heads=heads,
                    causal=rng.random() < 0.4)
    if kind in ("gru", "lstm"):
        return dict(kind=kind, dtype=rng.choice(["f32", "f32", "bf16", "f16"]), n=_log(rng, 2, 64), b=_log(rng, 1, 32),
                    t=_log(rng, 8, 128), i=_width(rng, 16, 256),
                    h=rng.choice([32, 50, 64, 96, 128, 128, 192, 256, 256, 384, 512]))
    return dict(kind="seq", dtype="bf16", n=_log(rng, 2, 64), b=_log(rng, 1, 16), t=_log(rng, 8, 128),
                v=_width(rng, 64, 8192), d=_width(rng, 32, 256), h=rng.choice([128, 256, 384, 512]))


def draw(rng):
    while True:
        c = _draw_one(rng)
        if c is None:
            continue
        w = work(c)
        flops, byts = _LIMITS[c["dtype"]]
        if c["kind"] == "seq":
            flops = 1.6e12
        if w["flops"] <= flops and w["bytes"] <= byts:
            return c


# ---------------------------------------------------------------------------------------
# models and inputs
# ---------------------------------------------------------------------------------------

def _out_hw(c):
    o = lambda s, k, p: (s + 2 * p - k) // c["stride"] + 1  # noqa: E731
    return (o(c["hh"], c["kh"], c["pad"]) if c["hh"] else 1), o(c["ww"], c["kw"], c["pad"])


def _modules(c):
    """The N torch models of a case (random default initialisation), on the GPU, in its dtype."""
    from wide_compiler.workloads import MLP, ResBlock, SeqModel
    n, kind, dt = c["n"], c["kind"], DTYPES[c["dtype"]]
    # cuDNN-style weight flattening of the torch recurrent modules is of no use here
    with torch.device(DEV), torch.backends.cudnn.flags(enabled=False), torch.no_grad():
        if kind == "mlp":
            mods = [MLP(c["i"], c["h"], c["o"]) for _ in range(n)]
        elif kind == "linear":
            mods = [nn.Linear(c["i"], c["o"], bias=c["bias"]) for _ in range(n)]
        elif kind == "layernorm":
            mods = [nn.LayerNorm(c["d"]) for _ in range(n)]
            for m in mods:
                m.weight.normal_(1.0, 0.1)
                m.bias.normal_(0.0, 0.1)
        elif kind == "conv":
            if c["hh"]:
                mods = [nn.Conv2d(c["ci"], c["co"], (c["kh"], c["kw"]), stride=c["stride"], padding=c["pad"])
                        for _ in range(n)]
            else:
                mods = [nn.Conv1d(c["ci"], c["co"], c["kw"], stride=c["stride"], padding=c["pad"]) for _ in range(n)]
        elif kind == "resblock":
            mods = [ResBlock(c["c"]) for _ in range(n)]
            for m in mods:
                for bn in (m.bn1, m.bn2):
                    bn.weight.normal_(1.0, 0.1)
                    bn.bias.normal_(0.0, 0.1)
                    bn.running_mean.normal_(0.0, 0.1)
                    bn.running_var.uniform_(0.5, 1.5)
        elif kind == "attention":
            mods = [nn.MultiheadAttention(c["d"], c["heads"], batch_first=True) for _ in range(n)]
            for m in mods:
                m.in_proj_bias.uniform_(-0.1, 0.1)
                m.out_proj.bias.uniform_(-0.1, 0.1)
        elif kind == "gru":
            mods = [nn.GRU(c["i"], c["h"], batch_first=True) for _ in range(n)]
        elif kind == "lstm":
            mods = [nn.LSTM(c["i"], c["h"], batch_first=True) for _ in range(n)]
        else:
            mods = [SeqModel(c["v"], c["d"], c["h"]) for _ in range(n)]
        return [m.to(dt).eval() for m in mods]


def _input(c):
    n, kind, dt = c["n"], c["kind"], DTYPES[c["dtype"]]
    if kind == "seq":
        return torch.randint(0, c["v"], (n, c["b"], c["t"]), device=DEV)
    shape = {
        "mlp": lambda: (c["b"], n * c["i"]),
        "linear": lambda: (n, c["b"], c["t"], c["i"]) if c["t"] else (n, c["b"], c["i"]),
        "layernorm": lambda: (n, c["b"], c["t"], c["d"]),
        "conv": lambda: (n, c["b"], c["ci"], c["hh"], c["ww"]) if c["hh"] else (n, c["b"], c["ci"], c["ww"]),
        "resblock": lambda: (c["b"], n * c["c"], c["hw"], c["hw"]),
        "attention": lambda: (n, c["b"], c["s"], c["d"]),
        "gru": lambda: (n, c["b"], c["t"], c["i"]),
        "lstm": lambda: (n, c["b"], c["t"], c["i"]),
    }[kind]()
    return torch.randn(shape, device=DEV).to(dt)


def prepare(case, seed):
    import wide_compiler as wc
    from wide_compiler.workloads import WideSeqModel
    c, kind = case, case["kind"]
    torch.manual_seed(seed)
    mods = _modules(c)
    x = _input(c)
    if kind == "mlp":
        wide = wc.compile(mods, x[:, :c["i"]].contiguous()).eval()
    elif kind == "resblock":
        wide = wc.compile(mods, x[:, :c["c"]].contiguous()).eval()
    elif kind == "seq":
        wide = WideSeqModel(mods).eval()
    else:
        cls = {"linear": wc.WideLinear, "layernorm": wc.WideLayerNorm, "attention": wc.WideAttention,
               "gru": wc.WideGRU, "lstm": wc.WideLSTM}.get(kind) or (wc.WideConv2d if c["hh"] else wc.WideConv1d)
        wide = cls.from_modules(mods).eval()
    return {"wide": wide, "x": x, "causal": bool(c.get("causal", False)), "kind": kind}


def run(state):
    with torch.no_grad():
        if state["kind"] == "attention":
            return state["wide"](state["x"], is_causal=state["causal"])
        if state["kind"] == "gru":
            out, h_n = state["wide"](state["x"])
            return [out, h_n]
        if state["kind"] == "lstm":
            out, (h_n, c_n) = state["wide"](state["x"])
            return [out, h_n, c_n]
        return state["wide"](state["x"])


# ---------------------------------------------------------------------------------------
# what a pass cannot do without, and how exactly it is computed
# ---------------------------------------------------------------------------------------

def work(case):
    c, kind, n = case, case["kind"], case["n"]
    es = 4 if c["dtype"] == "f32" else 2
    if kind == "mlp":
        w = c["i"] * c["h"] + c["h"] + c["h"] * c["o"] + c["o"]
        return {"bytes": es * n * (w + c["b"] * (c["i"] + c["o"])),
                "flops": 2 * n * c["b"] * (c["i"] * c["h"] + c["h"] * c["o"])}
    if kind == "linear":
        rows = c["b"] * max(c["t"], 1)
        return {"bytes": es * n * (c["i"] * c["o"] + c["o"] * c["bias"] + rows * (c["i"] + c["o"])),
                "flops": 2 * n * rows * c["i"] * c["o"]}
    if kind == "layernorm":
        e = n * c["b"] * c["t"] * c["d"]
        return {"bytes": es * (2 * e + 2 * n * c["d"]), "flops": 8 * e}
    if kind == "conv":
        ho, wo = _out_hw(c)
        taps = c["kh"] * c["kw"] * c["ci"]
        px = c["b"] * ho * wo
        return {"bytes": es * n * (c["co"] * (taps + 1) + c["b"] * c["ci"] * max(c["hh"], 1) * c["ww"] + px * c["co"]),
                "flops": 2 * n * px * c["co"] * taps}
    if kind == "resblock":
        px, ch = c["b"] * c["hw"] ** 2, c["c"]
        return {"bytes": es * n * (2 * (9 * ch * ch + 5 * ch) + 2 * px * ch), "flops": 4 * n * px * 9 * ch * ch}
    if kind == "attention":
        rows, d = n * c["b"] * c["s"], c["d"]
        keys = (c["s"] + 1) / 2 if c["causal"] else c["s"]
        return {"bytes": es * (n * (4 * d * d + 4 * d) + 2 * rows * d),
                "flops": int(8 * rows * d * d + 4 * rows * keys * d)}
    if kind in ("gru", "lstm"):
        g = (3 if kind == "gru" else 4) * c["h"]
        rows = n * c["b"] * c["t"]
        return {"bytes": es * (n * g * (c["i"] + c["h"] + 2) + rows * (c["i"] + c["h"]) + n * c["b"] * g),
                "flops": 2 * rows * g * (c["i"] + c["h"])}
    rows, g = n * c["b"] * c["t"], 4 * c["h"]
    used = n * min(c["v"], c["b"] * c["t"]) * c["d"]              # embedding rows that are looked up
    w = n * (g * (c["d"] + c["h"] + 2) + c["v"] * (c["h"] + 1) + 2 * c["d"])
    return {"bytes": 8 * rows + es * (used + w + rows * c["v"]),
            "flops": 2 * rows * (g * (c["d"] + c["h"]) + c["h"] * c["v"])}


def tolerance(case):
    return TOLERANCE[case["kind"]][case["dtype"]]


# About four times the largest difference from `exact` over the listed cases and 130 drawn ones.
# fp32: sums of a few hundred to a few thousand terms; 16-bit: the rounding of inputs, of
# intermediate tensors and of the result, which the recurrences carry through their steps.
TOLERANCE = {
    "mlp": {"f32": {"rel": 1.6e-6}, "bf16": {"rel": 1e-2}},
    "linear": {"f32": {"rel": 2.4e-6}, "bf16": {"rel": 7e-3}, "f16": {"rel": 8e-4}},
    "layernorm": {"f32": {"rel": 3e-7}, "bf16": {"rel": 7e-3}},
    "conv": {"f32": {"rel": 2e-6}, "bf16": {"rel": 7e-3}, "f16": {"rel": 8e-4}},
    "resblock": {"f32": {"rel": 1.5e-6}, "bf16": {"rel": 8e-3}},
    "attention": {"f32": {"rel": 2e-6}, "bf16": {"rel": 1.3e-2}, "f16": {"rel": 1.6e-3}},
    "gru": {"f32": {"rel": 1.5e-6}, "bf16": {"rel": 7e-3}, "f16": {"rel": 1.2e-3}},
    "lstm": {"f32": {"rel": 2e-6}, "bf16": {"rel": 9e-3}, "f16": {"rel": 1e-3}},
    "seq": {"bf16": {"rel": 1.2e-2}},
}


# ---------------------------------------------------------------------------------------
# the same forward in 64-bit torch
# ---------------------------------------------------------------------------------------

def _st(mods, name):
    """One parameter of all models in fp64, stacked: [N, ...]."""
    out = []
    for m in mods:
        v = m
        for part in name.split("."):
            v = getattr(v, part)
        out.append(v.detach())
    return torch.stack(out).double()


def _affine(x, w, b):
    """x [N, rows, K], w [N, O, K], b [N, O] or None."""
    y = torch.bmm(x, w.transpose(1, 2).contiguous())
    return y if b is None else y + b[:, None, :]


def _conv(x, w, b, stride, ph, pw):
    """x [N, B, Ci, H, W], w [N, Co, Ci, kh, kw], b [N, Co], model by model as a matrix product."""
    n, nb = x.shape[:2]
    kh, kw = w.shape[3:]
    ho, wo = (x.shape[3] + 2 * ph - kh) // stride + 1, (x.shape[4] + 2 * pw - kw) // stride + 1
    out = []
    for k in range(n):
        cols = nn.functional.unfold(x[k], (kh, kw), padding=(ph, pw), stride=stride)     # [B, Ci*kh*kw, L]
        out.append((torch.matmul(w[k].flatten(1), cols) + b[k][:, None]).reshape(nb, -1, ho, wo))
    return torch.stack(out)


def _norm(x, eps):
    mu = x.mean(-1, keepdim=True)
    return (x - mu) / ((x - mu).square().mean(-1, keepdim=True) + eps).sqrt()


def _recur(mods, kind, x, pre=""):
    """x [N, B, T, I] -> out [N, B, T, H] and the final state(s)."""
    w_ih, w_hh, b_ih, b_hh = (_st(mods, pre + k) for k in ("weight_ih_l0", "weight_hh_l0", "bias_ih_l0", "bias_hh_l0"))
    n, b, t, i = x.shape
    hid = w_hh.shape[2]
    gx = _affine(x.reshape(n, b * t, i), w_ih, b_ih).reshape(n, b, t, -1)
    w_t = w_hh.transpose(1, 2).contiguous()
    h = x.new_zeros(n, b, hid)
    cell = x.new_zeros(n, b, hid)
    out = x.new_empty(n, b, t, hid)
    for s in range(t):
        gh = torch.bmm(h, w_t) + b_hh[:, None, :]
        if kind == "gru":
            xr, xz, xn = gx[:, :, s].chunk(3, -1)
            hr, hz, hn = gh.chunk(3, -1)
            z = torch.sigmoid(xz + hz)
            h = (1 - z) * torch.tanh(xn + torch.sigmoid(xr + hr) * hn) + z * h
        else:
            gi, gf, gg, go = (gx[:, :, s] + gh).chunk(4, -1)
            cell = torch.sigmoid(gf) * cell + torch.sigmoid(gi) * torch.tanh(gg)
            h = torch.sigmoid(go) * torch.tanh(cell)
        out[:, :, s] = h
    return (out, h) if kind == "gru" else (out, h, cell)


def exact(case, seed):
    c, kind, n = case, case["kind"], case["n"]
    torch.manual_seed(seed)
    mods = _modules(c)
    with torch.no_grad():
        return _exact(c, kind, n, mods, _input(c))


def _exact(c, kind, n, mods, x):
    b = c["b"]
    if kind == "seq":
        emb = _st(mods, "emb.weight")
        h = torch.stack([emb[k][x[k]] for k in range(n)])
        del emb
        h = _norm(h, mods[0].ln.eps) * _st(mods, "ln.weight")[:, None, None, :] + _st(mods, "ln.bias")[:, None, None, :]
        h = _recur(mods, "lstm", h, "lstm.")[0].reshape(n, -1, c["h"])
        y = _affine(h, _st(mods, "fc.weight"), _st(mods, "fc.bias"))
        return y.reshape(n, b, c["t"], c["v"])
    x = x.double()
    if kind == "mlp":
        h = x.reshape(b, n, c["i"]).movedim(1, 0).contiguous()
        h = torch.relu(_affine(h, _st(mods, "fc1.weight"), _st(mods, "fc1.bias")))
        y = _affine(h, _st(mods, "fc2.weight"), _st(mods, "fc2.bias"))
        return y.movedim(0, 1).reshape(b, n * c["o"])
    if kind == "linear":
        y = _affine(x.reshape(n, -1, c["i"]), _st(mods, "weight"), _st(mods, "bias") if c["bias"] else None)
        return y.reshape(*x.shape[:-1], c["o"])
    if kind == "layernorm":
        return _norm(x, mods[0].eps) * _st(mods, "weight")[:, None, None, :] + _st(mods, "bias")[:, None, None, :]
    if kind == "conv":
        w, bias = _st(mods, "weight"), _st(mods, "bias")
        if c["hh"]:
            return _conv(x, w, bias, c["stride"], c["pad"], c["pad"])
        return _conv(x[:, :, :, None], w[:, :, :, None], bias, c["stride"], 0, c["pad"])[:, :, :, 0]
    if kind == "resblock":
        def bn(v, name):
            m, s = _st(mods, name + ".running_mean"), (_st(mods, name + ".running_var") + mods[0].bn1.eps).sqrt()
            shape = (n, 1, c["c"], 1, 1)
            return ((v - m.view(shape)) / s.view(shape) * _st(mods, name + ".weight").view(shape)
                    + _st(mods, name + ".bias").view(shape))
        h = x.reshape(b, n, c["c"], c["hw"], c["hw"]).movedim(1, 0).contiguous()
        y = torch.relu(bn(_conv(h, _st(mods, "conv1.weight"), _st(mods, "conv1.bias"), 1, 1, 1), "bn1"))
        y = bn(_conv(y, _st(mods, "conv2.weight"), _st(mods, "conv2.bias"), 1, 1, 1), "bn2")
        return torch.relu(y + h).movedim(0, 1).reshape(x.shape)
    if kind == "attention":
        s, d, heads = c["s"], c["d"], c["heads"]
        qkv = _affine(x.reshape(n, b * s, d), _st(mods, "in_proj_weight"), _st(mods, "in_proj_bias"))
        q, k, v = (t.reshape(n * b, s, heads, d // heads).transpose(1, 2).reshape(-1, s, d // heads)
                   for t in qkv.chunk(3, -1))
        a = torch.bmm(q, k.transpose(1, 2).contiguous()) * (d // heads) ** -0.5
        if c["causal"]:
            a = a.masked_fill(torch.ones(s, s, dtype=torch.bool, device=x.device).triu(1), float("-inf"))
        y = torch.bmm(torch.softmax(a, -1), v).reshape(n * b, heads, s, d // heads).transpose(1, 2)
        y = _affine(y.reshape(n, b * s, d), _st(mods, "out_proj.weight"), _st(mods, "out_proj.bias"))
        return y.reshape(n, b, s, d)
    r = _recur(mods, kind, x)
    return list(r)
