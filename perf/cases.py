"""The workloads this library's speed is judged by, each through a public entry point.

Five kinds of call, over the sizes users bring:

  ffn      moe_forward on a pure-NF4 rank-256 layer held in the tile layout:
           decode from one token up, prefill up to 4096 tokens, both output
           modes, bf16 / f16 / f32 activations
  hetero   moe_forward on a layer with per-expert ranks and INT8 groups
           (row layout), slots below a weight threshold dropped
  rows     moe_forward on a pure-NF4 layer of another rank (row layout)
  stack    DecodeStack: routers, expert FFNs and residual adds of consecutive
           layers replayed from one HIP graph
  router   Router: logits, softmax, top-k, renormalise
  expert   swiglu_expert: one expert, host arrays in and out

Weights are drawn with the spectrum of a factorized layer (rank component i
scaled by sqrt(s_i), s_i = 8 * i^-0.7, so gate pre-activations are a few
tenths) and packed here in plain torch; `exact` decodes the same packed bytes
and evaluates the chain in float64.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import latent_amd
from latent_amd.moe import DeviceFactor, StackedLayer
from latent_amd.router import Router
from latent_amd.runtime import load_pair, swiglu_expert
from latent_amd.stack import DecodeStack

# The NF4 levels of the packed format.
LEVELS = (-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635,
          -0.18477343022823334, -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725,
          0.24611230194568634, 0.33791524171829224, 0.44070982933044434, 0.5626170039176941,
          0.7229568362236023, 1.0)
GROUP = 32
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
RANKS = (64, 128, 256, 512)
BIG = {"E": 256, "d": 7168, "ff": 2048, "k": 8}


def listed():
    return [
        # One user's decode step: latency.
        dict(name="decode_1", kind="ffn", T=1, x="bf16", w="f32", slots=False, skew=0.0, R=256, **BIG),
        # A few concurrent users.
        dict(name="decode_8", kind="ffn", T=8, x="bf16", w="f32", slots=False, skew=0.0, R=256, **BIG),
        # A busy server's decode batch: almost every expert is read.
        dict(name="decode_64", kind="ffn", T=64, x="bf16", w="f32", slots=False, skew=0.0, R=256, **BIG),
        # A short prompt (or a chunk of one) through the ggml op's operands:
        # f16 activations and weights, unweighted per-slot output.
        dict(name="prompt_301_slots", kind="ffn", T=301, x="f16", w="f16", slots=True, skew=0.0, R=256, **BIG),
        # A long prompt with uneven expert popularity (about 5 to 430 tokens each).
        dict(name="prefill_4096", kind="ffn", T=4096, x="bf16", w="f32", slots=False, skew=1.5, R=256, **BIG),
        # A layer compressed by energy: ranks 64..512, a tenth of the groups
        # INT8, light slots dropped; a decode batch and a batched short prompt.
        dict(name="hetero_16", kind="hetero", T=16, x="bf16", R=512, **BIG),
        dict(name="hetero_256", kind="hetero", T=256, x="bf16", R=512, **BIG),
        # A smaller model at rank 128: decode batch and prompt.
        dict(name="rank128_24", kind="rows", T=24, x="bf16", E=64, d=2048, ff=1408, k=6, R=128),
        dict(name="rank128_1999", kind="rows", T=1999, x="bf16", E=64, d=2048, ff=1408, k=6, R=128),
        # A decode step of consecutive layers from one graph.
        dict(name="stack_32", kind="stack", T=32, layers=3, R=256, **BIG),
        # Routing of a long prompt.
        dict(name="router_4096", kind="router", T=4096, x="bf16", w="f32", E=256, d=7168, k=8),
        # One small expert from its stored artifacts, numpy in and out.
        dict(name="expert_4", kind="expert", T=4, q="nf4", d=512, ff=1408, R=64),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choices(("ffn", "hetero", "rows", "stack", "router", "expert"), (5, 2, 2, 1, 1, 1))[0]
    x = rng.choice(("bf16", "bf16", "f16", "f32"))
    if kind == "ffn":
        T = _log(rng, 1, 4096)
        slots = T <= 1024 and rng.random() < 0.3
        return dict(kind=kind, T=T, x=x, w=rng.choice(("f32", "f16")), slots=slots,
                    skew=rng.choice((0.0, round(rng.uniform(0.2, 1.5), 2))), R=256, **BIG)
    if kind == "hetero":
        return dict(kind=kind, T=_log(rng, 1, 256), x=x, R=512, **BIG)
    if kind == "rows":
        E, k = rng.choice(((16, 4), (64, 6), (128, 8)))
        return dict(kind=kind, T=_log(rng, 1, 2048), x=x, E=E, d=rng.choice((1024, 2048, 4096)),
                    ff=rng.choice((512, 1408, 2048)), k=k, R=rng.choice((64, 128, 192)))
    if kind == "stack":
        return dict(kind=kind, T=_log(rng, 1, 64), layers=rng.choice((2, 3)), R=256, **BIG)
    if kind == "router":
        E, k, d = rng.choice(((256, 8, 7168), (64, 6, 2048), (160, 6, 5120)))
        return dict(kind=kind, T=_log(rng, 1, 4096), x=x, w=rng.choice(("f32", "bf16")), E=E, d=d, k=k)
    return dict(kind=kind, T=_log(rng, 1, 16), q=rng.choice(("nf4", "int8")), d=rng.randrange(256, 1025, 8),
                ff=rng.randrange(352, 2817, 8), R=rng.randrange(32, 129, 4))


# ---- inputs ---------------------------------------------------------------------
def _gen(seed, tag=0):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1009 + tag)


def _levels(dtype):
    return torch.tensor(LEVELS, dtype=dtype, device="cuda")


def _nf4(v):
    """Codes u8 [..., cols/2] and scales f16 [..., cols/32] of f32 v [..., cols]."""
    lv = _levels(torch.float32)
    g = v.reshape(-1, GROUP)
    s = g.abs().amax(1, keepdim=True)
    s = torch.where(s == 0, torch.ones_like(s), s)
    c = torch.bucketize(g / s, (lv[1:] + lv[:-1]) / 2, out_int32=True).to(torch.uint8)
    codes = c[:, 0::2] | (c[:, 1::2] << 4)
    return codes.reshape(*v.shape[:-1], -1), s.half().reshape(*v.shape[:-1], -1)


def _spectrum(R):
    return (8.0 * torch.arange(1, R + 1, device="cuda", dtype=torch.float32).pow(-0.7)).sqrt()


def _shapes(c):
    d, ff, R = c["d"], c["ff"], c["R"]
    return {"gate_a": (d, R), "gate_b": (R, ff), "up_a": (d, R), "up_b": (R, ff), "down_a": (ff, R), "down_b": (R, d)}


def _ranks(c, seed):
    """True rank of each expert: every listed rank equally often in a hetero layer."""
    if c["kind"] != "hetero":
        return torch.full((c["E"],), c["R"], dtype=torch.int64, device="cuda")
    r = torch.tensor(RANKS, device="cuda").repeat(-(-c["E"] // len(RANKS)))[:c["E"]]
    return r[torch.randperm(c["E"], generator=_gen(seed, 1), device="cuda")]


def _factors(c, seed):
    """name -> dict of the packed tensors in the stacked row layout."""
    E, R, root, ranks = c["E"], c["R"], _spectrum(c["R"]), _ranks(c, seed)
    out, step = {}, 32
    for n, (name, (rows, cols)) in enumerate(_shapes(c).items()):
        gen = _gen(seed, 10 + n)
        f = {"codes": torch.empty((E, rows, cols // 2), dtype=torch.uint8, device="cuda"),
             "scales": torch.empty((E, rows, cols // GROUP), dtype=torch.float16, device="cuda")}
        masks, data = [], []
        for e in range(0, E, step):
            r = ranks[e:e + step]
            v = torch.randn((len(r), rows, cols), generator=gen, device="cuda")
            live = (torch.arange(R, device="cuda") < r[:, None]) * root
            v *= (live[:, None, :] if name.endswith("_a") else live[:, :, None])
            v *= (rows if name.endswith("_a") else cols) ** -0.5
            codes, scales = _nf4(v)
            if c["kind"] == "hetero":
                g = v.view(len(r), rows, cols // GROUP, GROUP)
                top = g.abs().amax(-1)
                m = (torch.rand(top.shape, generator=gen, device="cuda") < 0.1) & (top > 0)
                sel, s = g[m], (top[m] / 127).half()
                scales[m] = s
                codes.view(len(r), rows, cols // GROUP, GROUP // 2)[m] = 0
                data.append((sel / (top[m] / 127)[:, None]).round().clamp(-127, 127).to(torch.int8))
                masks.append(m)
            f["codes"][e:e + step], f["scales"][e:e + step] = codes, scales
        if masks:
            f["mask"], f["data"] = torch.cat(masks), torch.cat(data)
        out[name] = f
    return out, ranks


def _int8_tables(mask):
    """(bitmap words as i32, index of each row's first flagged group)."""
    E, rows, groups = mask.shape
    words = -(-groups // 32)
    pad = torch.zeros((E, rows, words * 32), dtype=torch.bool, device="cuda")
    pad[..., :groups] = mask
    word = torch.zeros((E, rows, words), dtype=torch.int64, device="cuda")
    for b in range(32):
        word += pad.view(E, rows, words, 32)[..., b].to(torch.int64) << b
    word = torch.where(word >= 2 ** 31, word - 2 ** 32, word).to(torch.int32)
    n = mask.sum(-1).reshape(-1)
    return word.contiguous(), (n.cumsum(0) - n).to(torch.int32).reshape(E, rows).contiguous()


def _layer(c, seed):
    facs, ranks = _factors(c, seed)
    made = {}
    for name, f in facs.items():
        ext = (*_int8_tables(f["mask"]), f["data"]) if "mask" in f else (None, None, None)
        made[name] = DeviceFactor(f["codes"], f["scales"], *ext)
    return StackedLayer(**made, ranks=ranks.to(torch.int32)[:, None].repeat(1, 3).contiguous())


def _routing(c, seed):
    """ids i32 [T, k], weights [T, k] of a softmax router."""
    gen = _gen(seed, 3)
    logits = torch.randn((c["T"], c["E"]), generator=gen, device="cuda")
    if c["kind"] == "hetero":
        logits = logits * 2.0  # a peaked router: about a sixth of the slots fall below the threshold
    if c.get("skew"):
        rank = torch.randperm(c["E"], generator=gen, device="cuda").float()
        logits = logits - c["skew"] * rank / (c["E"] - 1)
    top, ids = torch.softmax(logits, 1).topk(c["k"], 1)
    w, ids = top / top.sum(1, keepdim=True), ids.to(torch.int32)
    if c["kind"] == "hetero":
        drop = w < 0.05
        w, ids = w.masked_fill(drop, 0.0), ids.masked_fill(drop, -1)
    return ids.contiguous(), w.to(DTYPES[c.get("w", "f32")]).contiguous()


def _x(c, seed):
    return torch.randn((c["T"], c["d"]), generator=_gen(seed, 2), device="cuda").to(DTYPES[c.get("x", "f32")])


def _router_weight(c, seed):
    w = torch.randn((c["d"], c["E"]), generator=_gen(seed, 4), device="cuda") * c["d"] ** -0.5
    return w.to(DTYPES[c.get("w", "f32")])


def _artifacts(c, seed):
    """name.side -> (flat data, scales, shape) of one expert, as the NPZ artifacts store them."""
    gen, root, out = _gen(seed, 5), _spectrum(c["R"]), {}
    for name, (n_in, n_out) in {"gate": (c["d"], c["ff"]), "up": (c["d"], c["ff"]), "down": (c["ff"], c["d"])}.items():
        for side in "ab":
            rows, cols = (n_in, c["R"]) if side == "a" else (c["R"], n_out)
            v = torch.randn((rows, cols), generator=gen, device="cuda")
            v = v * (root * rows ** -0.5 if side == "a" else root[:, None] * cols ** -0.5)
            group = 32 if c["q"] == "nf4" else 64
            v = torch.nn.functional.pad(v.reshape(-1), (0, -rows * cols % group))
            if c["q"] == "nf4":
                data, scales = (t.reshape(-1) for t in _nf4(v.view(1, -1)))
            else:
                top = v.view(-1, group).abs().amax(1, keepdim=True) / 127
                data = (v.view(-1, group) / top).round().clamp(-127, 127).to(torch.int8).reshape(-1)
                scales = top.half().reshape(-1)
            out[f"{name}.{side}"] = (data, scales, (rows, cols))
    return out


def prepare(case, seed):
    c = case
    if c["kind"] == "stack":
        layers = [_layer(c, seed * 7 + l) for l in range(c["layers"])]
        routers = [Router(_router_weight(c, seed * 7 + l), c["k"]) for l in range(c["layers"])]
        x0 = _x(c, seed)
        stack = DecodeStack(layers, routers, c["T"])
        stack.load(x0)
        stack.capture()
        return {"kind": "stack", "stack": stack, "x": x0}
    if c["kind"] == "router":
        router = Router(_router_weight(c, seed), c["k"])
        router.workspace(c["T"])
        return {"kind": "router", "router": router, "x": _x(c, seed),
                "logits": torch.empty((c["T"], c["E"]), device="cuda")}
    if c["kind"] == "expert":
        arrays = {}
        for key, (data, scales, shape) in _artifacts(c, seed).items():
            arrays[f"{key}.{c['q']}"] = data.cpu().numpy()
            arrays[f"{key}.scales"] = scales.cpu().numpy()
            arrays[f"{key}.shape"] = np.array(shape)
        pairs = [load_pair(arrays, n) for n in ("gate", "up", "down")]
        for p in pairs:
            for f in (p.a, p.b):
                f.to_device(torch.device("cuda", torch.cuda.current_device()))
        return {"kind": "expert", "x": _x(c, seed).cpu().numpy(), "pairs": pairs}
    layer = _layer(c, seed)
    layer.workspace(c["T"], c["k"])
    ids, w = _routing(c, seed)
    return {"kind": "moe", "layer": layer, "x": _x(c, seed), "ids": ids, "w": w, "mode": 1 if c.get("slots") else 0}


def run(state):
    s = state
    if s["kind"] == "moe":
        return latent_amd.moe_forward(s["x"], s["ids"], s["w"], s["layer"], out_mode=s["mode"])
    if s["kind"] == "stack":
        s["stack"].load(s["x"])
        out = s["stack"].replay()
        return {"x": out, "y": s["stack"].y, "logits": s["stack"].logits}
    if s["kind"] == "router":
        ids, w = s["router"](s["x"], logits_out=s["logits"])
        return {"ids": ids, "weights": w, "logits": s["logits"]}
    return swiglu_expert(s["x"], *s["pairs"])


# ---- what a pass cannot do without ---------------------------------------------------
def _pairs(c):
    return c["T"] * c["k"] * (0.83 if c["kind"] == "hetero" else 1.0)


def _experts(c):
    """Distinct experts a uniform routing reaches."""
    return c["E"] * (1.0 - (1.0 - 1.0 / c["E"]) ** _pairs(c))


def work(case):
    c = case
    size = {"f32": 4, "f16": 2, "bf16": 2}
    if c["kind"] == "router":
        n = c["T"] * c["E"]
        return {"bytes": c["T"] * c["d"] * size[c["x"]] + c["d"] * c["E"] * size[c["w"]] + 4 * n + 8 * c["T"] * c["k"],
                "flops": 2.0 * n * c["d"]}
    if c["kind"] == "expert":
        n = 3 * c["R"] * (c["d"] + c["ff"])
        per = 0.5 + 2 / 32 if c["q"] == "nf4" else 1 + 2 / 64
        return {"bytes": n * per + 8 * c["T"] * c["d"], "flops": 2.0 * n * c["T"]}
    rank = sum(RANKS) / len(RANKS) if c["kind"] == "hetero" else c["R"]
    n = 3 * rank * (c["d"] + c["ff"])
    per = 0.5 + 2 / 32 + (0.1 * 16 / 32 if c["kind"] == "hetero" else 0.0)
    one = _experts(c) * n * per + c["T"] * c["k"] * 8
    x, out = c["T"] * c["d"] * size[c.get("x", "f32")], 4 * c["T"] * c["d"] * (c["k"] if c.get("slots") else 1)
    flops = 2.0 * n * _pairs(c)
    if c["kind"] == "stack":
        rw = c["d"] * c["E"]
        return {"bytes": c["layers"] * (one + 4 * rw + out) + 2 * out, "flops": c["layers"] * (flops + 2.0 * c["T"] * rw)}
    return {"bytes": one + x + out, "flops": flops}


def tolerance(case):
    c = case
    if c["kind"] == "router":  # fp32 sums; ids may swap where two logits tie
        return {"rel": 1e-5, "differ": 1e-3}
    if c["kind"] == "expert":  # fp32 throughout
        return {"rel": 1e-5}
    pairs = c["T"] * c["k"]
    if c["kind"] == "hetero" and pairs < 16:
        return {"rel": 1e-5}
    if c["kind"] == "rows" and (pairs < 16 or 32 <= pairs <= 512) and pairs < 16 * c["E"]:
        return {"rel": 1e-5}
    # fp16 operands at each of the four products, fp32 sums: 3e-4 to 8e-4 off float64.
    return {"rel": 2e-3}


# ---- the same in float64 ------------------------------------------------------------
def _decode64(f, e):
    """f64 [rows, cols] of expert e."""
    codes = f["codes"][e].to(torch.int64)
    v = _levels(torch.float64)[torch.stack((codes & 15, codes >> 4), -1)]
    s = f["scales"][e].double()
    v = v.reshape(s.shape[0], s.shape[1], GROUP)
    if "mask" in f:
        n = int(f["mask"][:e].sum())
        m = f["mask"][e]
        v[m] = f["data"][n:n + int(m.sum())].double()
    return (v * s[..., None]).reshape(s.shape[0], -1)


def _swiglu64(x, a):
    g, u = x @ a[0] @ a[1], x @ a[2] @ a[3]
    return g * torch.sigmoid(g) * u @ a[4] @ a[5]


def _moe64(c, facs, x, ids, w, slots):
    y = torch.zeros((c["T"], c["k"], c["d"]) if slots else (c["T"], c["d"]), dtype=torch.float64, device="cuda")
    for e in torch.unique(ids).tolist():
        if e < 0:
            continue
        t, s = torch.nonzero(ids == e, as_tuple=True)
        v = _swiglu64(x[t], [_decode64(facs[n], e) for n in ("gate_a", "gate_b", "up_a", "up_b", "down_a", "down_b")])
        if slots:
            y[t, s] = v
        else:
            y.index_add_(0, t, v * w[t, s].double()[:, None])
    return y


def exact(case, seed):
    c = case
    if c["kind"] == "expert":
        mats = []
        for data, scales, (rows, cols) in _artifacts(c, seed).values():
            if c["q"] == "nf4":
                d = data.to(torch.int64)
                v = _levels(torch.float64)[torch.stack((d & 15, d >> 4), -1)].reshape(-1, 32)
            else:
                v = data.double().view(-1, 64)
            mats.append((v * scales.double()[:, None]).reshape(-1)[:rows * cols].view(rows, cols))
        return _swiglu64(_x(c, seed).double(), mats).cpu().numpy()
    x = _x(c, seed).double()
    if c["kind"] == "router":
        logits = x @ _router_weight(c, seed).double()
        top = logits.topk(c["k"], 1).values
        return {"ids": None, "weights": torch.softmax(top, 1), "logits": logits}
    if c["kind"] == "stack":
        ys, ls = [], []
        for l in range(c["layers"]):
            ls.append(x @ _router_weight(c, seed * 7 + l).double())
            top, ids = ls[-1].topk(c["k"], 1)
            ys.append(_moe64(c, _factors(c, seed * 7 + l)[0], x, ids, torch.softmax(top, 1), False))
            x = x + ys[-1]
        return {"x": x, "y": ys, "logits": ls}
    ids, w = _routing(c, seed)
    return _moe64(c, _factors(c, seed)[0], x, ids, w, bool(c.get("slots")))
