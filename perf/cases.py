"""The work that is timed: calls of the A81W41 layer, and prompts and decoding of the three model families.

Everything goes through the entry points that a user's program calls (``Linear``, ``Qwen3Model``, ``Model``).  Weights
are what such a program keeps: layers of one shape get them from the case's seed, a model is loaded once for each
configuration and serves every prompt (the seed draws the prompt).  A case is a dict of plain values:

  what "linear"    rows, out, in           one call of a layer
  what "row"       hidden, kv, ffn         the seven linears of a decoder layer for one token, at the grouped call sites
  what "prompt"    model, width, layers, tokens          a prompt, logits of its last token
  what "generate"  model, width, layers, tokens, new     a short prompt, then greedy tokens; logits behind them
  what "steps"     model, width, layers, tokens, new     a short prompt, then given tokens one call each, logits of each
"""
import json
import math
import os
import struct
import tempfile

import numpy as np
import torch

from __graft_entry__ import import_package

VOCAB = 32768
BLOCK = 32           # values that share a scale
HEAD = 128           # width of a head
WEIGHTS_SEED = 20    # of a model's weights: one checkpoint for all prompts


# ---- the cases -------------------------------------------------------------------------------

def listed():
    return [
        # one key projection of a decode step: the smallest call, launch and latency
        {"name": "k_proj 1 row", "what": "linear", "rows": 1, "out": 1024, "in": 4096},
        # what a decoder layer asks of the linears for one token
        {"name": "layer 1 row", "what": "row", "hidden": 4096, "kv": 1024, "ffn": 12288},
        # a handful of sequences decoded together, or a draft of five tokens checked
        {"name": "o_proj 5 rows", "what": "linear", "rows": 5, "out": 4096, "in": 4096},
        # a larger batch, and rows that fill no tile
        {"name": "down_proj 57 rows", "what": "linear", "rows": 57, "out": 4096, "in": 12288},
        # the prompt length the benchmark is quoted on, at the fused gate and up call site
        {"name": "gate_up 322 rows", "what": "linear", "rows": 322, "out": 24576, "in": 4096},
        # a long prompt
        {"name": "gate_proj 2047 rows", "what": "linear", "rows": 2047, "out": 12288, "in": 4096},
        # the forward pass around the layer at the 8B sizes (four of its layers): prompt, and an answer
        {"name": "qwen3 prompt", "what": "prompt", "model": "qwen3", "width": 4096, "layers": 4, "tokens": 322},
        {"name": "qwen3 answer", "what": "generate", "model": "qwen3", "width": 4096, "layers": 4, "tokens": 40, "new": 64},
        # the models with bfloat16 weights at the benchmark's 2k sizes: a long document, and an answer
        {"name": "takosun prompt", "what": "prompt", "model": "takosun", "width": 2048, "layers": 4, "tokens": 4095},
        {"name": "takosun answer", "what": "generate", "model": "takosun", "width": 2048, "layers": 4, "tokens": 33, "new": 64},
        {"name": "dimesun prompt", "what": "prompt", "model": "dimesun", "width": 2048, "layers": 2, "tokens": 2048},
        # a caller that samples by itself: one call and one row of logits a token
        {"name": "dimesun steps", "what": "steps", "model": "dimesun", "width": 2048, "layers": 2, "tokens": 33, "new": 32},
    ]


def _spread(rng, low, high, step=1):
    """A multiple of step, even over the logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high))) / step)) * step))


def draw(rng):
    if rng.random() < 0.5:
        return {"what": "linear", "rows": _spread(rng, 1, 2047), "out": _spread(rng, 512, 12288, 8), "in": _spread(rng, 512, 4096, 64)}
    if rng.random() < 0.15:
        return {"what": "row", "hidden": _spread(rng, 1024, 4096, 128), "kv": 128 * rng.randint(1, 8), "ffn": _spread(rng, 2048, 12288, 64)}
    model = rng.choice(["qwen3", "takosun", "dimesun"])
    case = {"model": model, "width": rng.choice([1024, 1536, 2048]), "layers": 2 if model == "dimesun" else rng.choice([2, 4])}
    if rng.random() < 0.6:
        return dict(case, what="prompt", tokens=_spread(rng, 16, 2048))
    what = "steps" if model == "dimesun" else rng.choice(["generate", "steps"])
    return dict(case, what=what, tokens=rng.randint(9, 99), new=rng.randint(8, 48))


# ---- A81W41 weights ---------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, device="cuda", generator=g).mul_(std)


def _quantize_weight(w):
    """fp32 [N][K] -> codes 0..15 [N][K], scale and minimum [N][K / 32] (binary16 values)."""
    b = w.view(w.shape[0], -1, BLOCK)
    low, high = b.amin(2), b.amax(2)
    scale, low = ((high - low) / 15).half().float(), low.half().float()
    codes = ((b - low[..., None]) / scale[..., None]).round_().clamp_(0, 15).to(torch.uint8)
    return codes.view(w.shape), scale, low


def _blobs(codes, scale, low):
    """The two packed forms of a weight (host bytes): blocks of 8 columns x 64 values with binary16 and with fp32 parameters."""
    groups, supers = codes.shape[0] // 8, codes.shape[1] // 64
    c = codes.view(groups, 8, supers, 2, 8, 4)
    q = (c[:, :, :, 0] | c[:, :, :, 1] << 4).permute(0, 2, 3, 1, 4).reshape(groups, supers, 256)
    params = torch.cat([p.view(groups, 8, supers, 2).permute(0, 2, 3, 1).reshape(groups, supers, 16) for p in (scale, low)], 2)
    return tuple(torch.cat([params.to(t).contiguous().view(torch.uint8), q], 2).cpu().numpy().reshape(-1) for t in (torch.float16, torch.float32))


def _layer_weight(g, out, k):
    return _quantize_weight(_normal(g, out, k, std=k ** -0.5))


def _activations(g, rows, k):
    """Normed activations: one channel in a thousand is large."""
    x = _normal(g, rows, k)
    x[:, torch.randperm(k, device="cuda", generator=g)[:max(1, k // 1000)]] *= 20.0
    return x


def _row_shapes(case):
    h, kv, f = case["hidden"], case["kv"], case["ffn"]
    return [("q", h, h), ("k", kv, h), ("v", kv, h), ("o", h, h), ("gate", f, h), ("up", f, h), ("down", h, f)]


# ---- models -----------------------------------------------------------------------------------
# A trained model's next token stands out; random weights leave thousands of close calls.  The head's row of token
# t + SHIFT is therefore the embedding of t, which the stream carries to the end.
SHIFT = 7919


def _qwen3_sizes(case):
    heads = case["width"] // HEAD
    return dict(n_layers=case["layers"], hidden=case["width"], n_q_heads=heads, n_kv_heads=max(1, heads // 4),
                intermediate=3 * case["width"], vocab=VOCAB, max_seq=2304)


def _qwen3_weights(case):
    """Yields (layer, what, value) in a fixed order; a linear's value is its codes, scale and minimum."""
    g, c = _generator(WEIGHTS_SEED), _qwen3_sizes(case)
    h, f, kv = c["hidden"], c["intermediate"], c["n_kv_heads"] * HEAD
    for i in range(c["n_layers"]):
        for which, (n, k) in enumerate([(h + 2 * kv, h), (h, h), (2 * f, h), (h, f)]):
            yield i, which, _layer_weight(g, n, k)
        yield i, "norms", [1.0 + _normal(g, n, std=0.1) for n in (h, h, HEAD, HEAD)]
    embed = _normal(g, VOCAB, h).half()
    yield -1, "embed", embed
    yield -1, "final", 1.0 + _normal(g, h, std=0.1)
    yield -1, 0, _quantize_weight(embed.float().roll(SHIFT, 0).mul_(h ** -0.5))


def _load_qwen3(pkg, case):
    model = pkg.Qwen3Model(**_qwen3_sizes(case))
    for i, what, value in _qwen3_weights(case):
        if what == "norms":
            for n, w in enumerate(value):
                model.set_norm(i, n, w.cpu().numpy())
        elif what == "final":
            model.set_norm(-1, 0, value.cpu().numpy())
        elif what == "embed":
            model.set_embedding(value.cpu().numpy())
        else:
            b16, b32 = _blobs(*value)
            model.set_linear_blobs(i, what, b16, b32 if i >= 0 else None)
    return model


def _takosun_config(case):
    w = case["width"]
    layers = []
    for i in range(case["layers"]):
        mixer = {"heads": w // HEAD, "dim": HEAD, "rot_dim": 64, "vdim": HEAD, "q_rank": w * 3 // 8, "kv_rank": 512, "scale": 192.0 ** -0.5,
                 "rot": {"base": 10000.0, "dims": 64}}
        if i % 2:
            mixer["kv_from"] = i - 1
        mlp = {"kind": "dense", "ff": 3 * w}
        if i == 1:
            mlp = {"kind": "moe", "router": {"experts": 16, "top": 4}, "expert": {"ff": w // 2}, "shared": {"ff": w // 2}}
        layers.append({"type": "latent_attention", "mixer": mixer, "mlp": mlp})
    return {"architecture": "Takosun", "vocab": VOCAB, "width": w, "norm": {"eps": 1e-6, "groups": 8}, "layers": layers}


def _dimesun_config(case):
    w = case["width"]
    mlp = {"kind": "moe", "router": {"experts": 32, "top": 4}, "expert": {"ff": w // 2, "limit": 7.0}}
    attention = {"heads": w // HEAD, "kv_heads": w // 512, "dim": HEAD, "vdim": HEAD, "rot": {"base": 10000.0, "dims": 64},
                 "mask": {"size": 1024}, "scale": HEAD ** -0.5}
    memory = {"heads": 8, "dim": w // 16, "vdim": w // 8, "gate_cap": 15.0}
    layers = [{"type": "mlstm", "mixer": memory, "mlp": mlp} if i % 2 else {"type": "attention", "mixer": attention, "mlp": mlp}
              for i in range(case["layers"])]
    return {"architecture": "Dimesun", "vocab": VOCAB, "width": w, "norm": {"eps": 1e-6}, "residual_mult": 0.5, "layers": layers,
            "loop": {"start": 0, "stop": case["layers"], "times": 2}}


def _config(case):
    return _takosun_config(case) if case["model"] == "takosun" else _dimesun_config(case)


def _dense_weights(case):
    """Tensors of the checkpoint by name, bfloat16 (tables int32), on the GPU."""
    g, cfg, w = _generator(WEIGHTS_SEED), _config(case), {}
    width = cfg["width"]

    def lin(name, n, k, gain=1.0):
        w[name] = _normal(g, n, k, std=gain * k ** -0.5).bfloat16()

    def vec(name, n, mean=1.0, std=0.1):
        w[name] = (mean + _normal(g, n, std=std)).bfloat16()

    def ff(prefix, n):
        lin(prefix + "gate", n, width)
        lin(prefix + "up", n, width)
        lin(prefix + "down", width, n)

    w["embed"] = _normal(g, VOCAB, width).bfloat16()
    for i, layer in enumerate(cfg["layers"]):
        p, m, f = f"l{i}.", layer["mixer"], layer["mlp"]
        mix, mlp = p + "mix.", p + "mlp."
        if layer["type"] == "latent_attention":
            heads, dim, rot, vdim, rank = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
            for n, mean in (("norm1", 1.0), ("norm1b", 0.3), ("norm2", 1.0), ("norm2b", 0.3)):
                vec(p + n, width, mean)
            lin(mix + "dq", m["q_rank"], width)
            vec(mix + "dq.norm", m["q_rank"])
            lin(mix + "uq", heads * (dim + rot), m["q_rank"], 1.5)
            if "kv_from" not in m:
                lin(mix + "dkv", rank + rot, width)
                vec(mix + "dkv.norm", rank)
            lin(mix + "uk", heads * dim, rank, 1.5)
            lin(mix + "uv", heads * vdim, rank)
            lin(mix + "g", heads, width)
            lin(mix + "o", width, heads * vdim)
            if f["kind"] == "dense":
                ff(mlp, f["ff"])
            else:
                experts, top = f["router"]["experts"], f["router"]["top"]
                for e in range(experts):
                    ff(mlp + f"e{e}.", f["expert"]["ff"])
                w[mlp + "table"] = torch.rand(VOCAB, experts, device="cuda", generator=g).argsort(1)[:, :top].int().contiguous()
                ff(mlp + "shared.", f["shared"]["ff"])
            vec(p + "dwa", i + 2, 0.0)
            w[p + "dwa"][-1] += 1.0
            continue
        vec(p + "norm1", width, 0.0)
        heads, dim, vdim = m["heads"], m["dim"], m["vdim"]
        if layer["type"] == "mlstm":
            lin(mix + "q", heads * dim, width, 1.5)
            lin(mix + "k", heads * dim, width)
            w[mix + "k"] = (0.7 * w[mix + "k"].float() + 0.5 * w[mix + "q"].float()).bfloat16()  # a key resembles its query
            lin(mix + "v", heads * vdim, width)
            lin(mix + "g", heads * vdim, width)
            lin(mix + "i", heads, width)
            vec(mix + "i.b", heads, 0.0, 1.0)
            lin(mix + "f", heads, width)
            vec(mix + "f.b", heads, 3.0, 2.0)  # some heads remember for long, some forget soon
            vec(mix + "norm", heads * vdim)
        else:
            lin(mix + "q", heads * dim, width, 1.5)
            lin(mix + "k", m["kv_heads"] * dim, width, 1.5)
            lin(mix + "v", m["kv_heads"] * vdim, width)
        lin(mix + "o", width, heads * vdim)
        lin(mlp + "router", f["router"]["experts"], width, 2.0)
        vec(mlp + "router.b", f["router"]["experts"], 0.0, 0.5)
        for e in range(f["router"]["experts"]):
            ff(mlp + f"e{e}.", f["expert"]["ff"])
    if "loop" in cfg:
        w["loop.step"] = _normal(g, cfg["loop"]["times"], width, std=0.3).bfloat16()
        vec("final.norm", width, 0.0)
    else:
        vec("final.norm", width)
        w["head"] = (w["embed"].float().roll(SHIFT, 0) * width ** -0.5).bfloat16()
    return w


def _load_dense(pkg, case):
    """Through the checkpoint format: config.json and model.safetensors."""
    header, raws, at = {}, [], 0
    for name, t in _dense_weights(case).items():
        raw = t.cpu().view(torch.int32 if t.dtype == torch.int32 else torch.int16).numpy()
        header[name] = {"dtype": "I32" if t.dtype == torch.int32 else "BF16", "shape": list(t.shape), "data_offsets": [at, at + raw.nbytes]}
        raws.append(raw)
        at += raw.nbytes
    with tempfile.TemporaryDirectory() as root:
        with open(os.path.join(root, "config.json"), "w") as f:
            json.dump(_config(case), f)
        text = json.dumps(header).encode()
        with open(os.path.join(root, "model.safetensors"), "wb") as f:
            f.write(struct.pack("<Q", len(text)) + text)
            for raw in raws:
                raw.tofile(f)
        return pkg.Model.load(root, 4352)


_models = {}  # a program loads a model once and gives it one prompt after the other


def _model(case):
    key = (case["model"], case["width"], case["layers"])
    if key not in _models:
        _models[key] = (_load_qwen3 if case["model"] == "qwen3" else _load_dense)(import_package(), case)
    return _models[key]


def _tokens(case, seed):
    return np.random.default_rng(seed).integers(0, VOCAB, case["tokens"] + case.get("new", 0)).astype(np.int32)


# ---- measured calls ---------------------------------------------------------------------------

def prepare(case, seed):
    if case["what"] in ("prompt", "generate", "steps"):
        return {"what": case["what"], "model": _model(case), "ids": _tokens(case, seed), "prompt": case["tokens"], "new": case.get("new", 0)}
    pkg, g = import_package(), _generator(seed)
    shapes = [("", case["out"], case["in"])] if case["what"] == "linear" else _row_shapes(case)
    layers = {name: pkg.Linear.from_blobs(*_blobs(*_layer_weight(g, n, k)), n, k) for name, n, k in shapes}
    if case["what"] == "linear":
        return {"what": "linear", "layer": layers[""], "x": _activations(g, case["rows"], case["in"])}
    return {"what": "row", "layers": layers, "x": _activations(g, 1, case["hidden"]), "attention": _normal(g, 1, case["hidden"]),
            "h": _activations(g, 1, case["hidden"]), "act": _normal(g, 1, case["ffn"])}


def run(state):
    what = state["what"]
    if what == "linear":
        return state["layer"].forward(state["x"])
    if what == "row":
        n = state["layers"]
        multi = n["q"].forward_multi
        return (multi([n["q"], n["k"], n["v"]], state["x"]) + [n["o"].forward(state["attention"])]
                + multi([n["gate"], n["up"]], state["h"]) + [n["down"].forward(state["act"])])
    model, ids, prompt = state["model"], state["ids"], state["prompt"]
    model.reset()
    if what == "prompt":
        return model.forward(ids)
    if what == "generate":
        tokens, _, _ = model.generate_greedy(ids[:prompt], state["new"])
        return tokens, model.forward(tokens[-1:])
    return [model.forward(ids[:prompt])] + [model.forward(ids[i:i + 1]) for i in range(prompt, len(ids))]


# ---- what a pass cannot do without ------------------------------------------------------------

def _linear_work(rows, n, k):
    return 0.625 * n * k + 4.0 * rows * (k + n), 2.0 * rows * n * k


def _model_sizes(case, tokens):
    """Weights a pass over `tokens` new tokens reads, weights each token meets, multiply-adds of attention over `keys` keys."""
    w = case["width"]
    if case["model"] == "qwen3":
        c = _qwen3_sizes(case)
        kv = c["n_kv_heads"] * HEAD
        per = (w + 2 * kv) * w + w * w + 9 * w * w
        return c["n_layers"] * per, c["n_layers"] * per, c["n_layers"] * 2 * w, 0
    cfg, once, each, attention, states = _config(case), 0, 0, 0, 0
    times = cfg.get("loop", {"times": 1})["times"]
    for layer in cfg["layers"]:
        m, f = layer["mixer"], layer["mlp"]
        if layer["type"] == "latent_attention":
            mix = w * (m["q_rank"] + m["heads"] + (0 if "kv_from" in m else m["kv_rank"] + m["rot_dim"]))
            mix += m["q_rank"] * m["heads"] * (m["dim"] + m["rot_dim"]) + m["heads"] * (m["dim"] + m["vdim"]) * m["kv_rank"]
            mix += w * m["heads"] * m["vdim"]
            attention += m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
        elif layer["type"] == "mlstm":
            mix = w * m["heads"] * (2 * m["dim"] + 3 * m["vdim"] + 2)
            states += m["heads"] * m["dim"] * m["vdim"]
        else:
            mix = w * (2 * m["heads"] * m["dim"] + m["kv_heads"] * (m["dim"] + m["vdim"]))
            attention += 2 * m["heads"] * m["dim"]
        if f["kind"] == "dense":
            once, each = once + mix + 3 * w * f["ff"], each + mix + 3 * w * f["ff"]
            continue
        expert, experts, top = 3 * w * f["expert"]["ff"], f["router"]["experts"], f["router"]["top"]
        shared = 3 * w * f["shared"]["ff"] if "shared" in f else w * experts
        each += mix + top * expert + shared
        once += mix + min(experts, top * tokens) * expert + shared
    return once * times, each * times, attention * times, states * times


def _pass_work(case, before, tokens):
    """One pass over `tokens` new tokens on top of `before`, logits of the last one."""
    once, each, attention, states = _model_sizes(case, tokens)
    size = 0.625 if case["model"] == "qwen3" else 2.0
    keys = tokens * before + tokens * (tokens + 1) / 2
    if case["model"] == "dimesun":
        keys = sum(p % 1024 + 1 for p in range(before, before + tokens))
    nbytes = size * (once + VOCAB * case["width"]) + 4.0 * VOCAB + 8.0 * states
    return nbytes, 2.0 * (each * tokens + VOCAB * case["width"] + attention * keys + 2 * states * tokens)


def work(case):
    if case["what"] == "linear":
        parts = [_linear_work(case["rows"], case["out"], case["in"])]
    elif case["what"] == "row":
        parts = [_linear_work(1, n, k) for _, n, k in _row_shapes(case)]
    else:
        parts = [_pass_work(case, 0, case["tokens"])] + [_pass_work(case, case["tokens"] + i, 1) for i in range(case.get("new", 0))]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    # Four times what was seen between two of the framework's own paths on the same inputs.  Linears: int8 against
    # block-scaled matrix ops (6e-6, at most 5e-5 of a value).  Models: other attention kernels, other one-token kernels (Qwen3
    # 0.012, whose activations are rounded to 8 bits before every linear; Takosun 0.009; Dimesun 0.004).
    if case["what"] in ("linear", "row"):
        return {"rel": 2.5e-5, "max": 2e-4}
    if case["model"] == "dimesun":
        return {"rel": 0.015, "max": 0.07}
    return {"rel": 0.03, "max": 0.2}


# ---- the same in 64 bits ----------------------------------------------------------------------

def _quantized_rows(x, half):
    """What the layer contracts: the rows' quantised values times their scale, and per 32 the scaled sum."""
    b = x.float().view(x.shape[0], -1, BLOCK)
    amax = b.abs().amax(2)
    # IEEE quotients in 32 bits: torch multiplies by a rounded reciprocal there
    d, inv = (amax.double() / 127.0).float(), (127.0 / amax.double()).float()
    inv = torch.where(amax != 0, inv, torch.zeros_like(inv))
    q = (b * inv[..., None]).round().clamp_(-128, 127)
    sums = d * q.sum(2)
    if half:
        d, sums = d.half().float(), sums.half().float()
    return (q.double() * d.double()[..., None]).view(x.shape), sums.double()


def _linear_exact(weight, x, half=None):
    codes, scale, low = weight
    rows, sums = _quantized_rows(x, x.shape[0] == 1 if half is None else half)
    out = torch.empty(x.shape[0], codes.shape[0], dtype=torch.float64, device="cuda")
    for n0 in range(0, codes.shape[0], 4096):
        part = slice(n0, min(n0 + 4096, codes.shape[0]))
        w = codes[part].double().view(-1, scale.shape[1], BLOCK) * scale[part].double()[..., None]
        out[:, part] = rows @ w.view(-1, codes.shape[1]).t() + sums @ low[part].double().t()
    return out


def _rms(x, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)


def _rotate(x, positions, base):
    """Component i of the last axis turns with component i + half; x [T][...][dims]."""
    half = x.shape[-1] // 2
    freq = base ** (-2.0 * torch.arange(half, dtype=torch.float64, device="cuda") / x.shape[-1])
    angle = positions.double()[:, None] * freq
    angle = angle.view((len(positions),) + (1,) * (x.dim() - 2) + (half,))
    c, s, u, v = angle.cos(), angle.sin(), x[..., :half], x[..., half:]
    return torch.cat([u * c - v * s, v * c + u * s], -1)


def _mask(positions, keys, chunk=None):
    t, s = positions[:, None], keys[None, :]
    return (s <= t) if chunk is None else (s <= t) & (s // chunk == t // chunk)


class _Qwen3Exact:
    """Keys and values are kept as the framework keeps them (binary16); a single row is quantised with binary16 scales."""

    def __init__(self, case):
        self.c = _qwen3_sizes(case)
        self.lin, self.norms, self.kept, self.at = {}, {}, {}, 0
        for i, what, value in _qwen3_weights(case):
            if what == "norms":
                self.norms[i] = [v.double() for v in value]
            elif what == "final":
                self.final = value.double()
            elif what == "embed":
                self.embed = value
            else:
                self.lin[i, what] = value

    def forward(self, ids):
        c, n = self.c, len(ids)
        heads, kv = c["n_q_heads"], c["n_kv_heads"]
        at = torch.arange(self.at, self.at + n, device="cuda")
        x = self.embed[torch.as_tensor(np.asarray(ids), device="cuda").long()].double()
        for i in range(c["n_layers"]):
            w = self.norms[i]
            qkv = _linear_exact(self.lin[i, 0], _rms(x, 1e-6) * w[0])
            q, k, v = qkv.split([heads * HEAD, kv * HEAD, kv * HEAD], 1)
            q = _rotate(_rms(q.view(n, heads, HEAD), 1e-6) * w[2], at, 1e6)
            k = _rotate(_rms(k.view(n, kv, HEAD), 1e-6) * w[3], at, 1e6).half().double()
            v = v.reshape(n, kv, HEAD).half().double()
            if i in self.kept:
                k, v = torch.cat([self.kept[i][0], k]), torch.cat([self.kept[i][1], v])
            self.kept[i] = k, v
            sees = _mask(at, torch.arange(len(k), device="cuda"))
            out = [(q[:, a] @ k[:, a * kv // heads].t() * HEAD ** -0.5).masked_fill(~sees, -math.inf).softmax(1) @ v[:, a * kv // heads]
                   for a in range(heads)]
            x = x + _linear_exact(self.lin[i, 1], torch.cat(out, 1))
            gate, up = _linear_exact(self.lin[i, 2], _rms(x, 1e-6) * w[1]).chunk(2, 1)
            x = x + _linear_exact(self.lin[i, 3], gate * gate.sigmoid() * up)
        self.at += n
        return _linear_exact(self.lin[-1, 0], (_rms(x, 1e-6) * self.final)[-1:], half=True)[0]


class _DenseExact:
    """A sequence from its start: logits at the last `want` tokens."""

    def __init__(self, case):
        self.cfg, self.w = _config(case), _dense_weights(case)

    def lin(self, x, name):
        return x @ self.w[name].double().t()

    def expert_sum(self, h, chosen, weights, one):
        out = torch.zeros_like(h)
        for e in range(int(chosen.max()) + 1):
            token, slot = (chosen == e).nonzero(as_tuple=True)
            if len(token):
                out.index_add_(0, token, one(h[token], e) * weights[token, slot][:, None])
        return out

    def forward(self, ids, want):
        ids = torch.as_tensor(np.asarray(ids), device="cuda").long()
        at = torch.arange(len(ids), device="cuda")
        x = (self.takosun if "loop" not in self.cfg else self.dimesun)(ids, at)
        return x[len(ids) - want:] @ self.w["embed" if "loop" in self.cfg else "head"].double().t()

    def takosun(self, ids, at):
        cfg, w, n = self.cfg, self.w, len(ids)
        eps, groups, width = cfg["norm"]["eps"], cfg["norm"]["groups"], cfg["width"]

        def norm(v, name):
            return _rms(v.view(n, groups, width // groups), eps).view(n, width) * w[name].double()

        def ff(h, prefix):
            gate = self.lin(h, prefix + "gate")
            return self.lin(gate * gate.sigmoid() * self.lin(h, prefix + "up"), prefix + "down")

        x = w["embed"][ids].double()
        states, latents, sees = [x], {}, _mask(at, at)
        for i, layer in enumerate(cfg["layers"]):
            p, m, f = f"l{i}.", layer["mixer"], layer["mlp"]
            mix, mlp = p + "mix.", p + "mlp."
            heads, dim, base = m["heads"], m["dim"], m["rot"]["base"]
            h = norm(x, p + "norm1")
            if "kv_from" not in m:
                both = self.lin(h, mix + "dkv")
                latents[i] = (_rms(both[:, :m["kv_rank"]], eps) * w[mix + "dkv.norm"].double(), _rotate(both[:, m["kv_rank"]:], at, base))
            latent, k_rot = latents[m.get("kv_from", i)]
            q = self.lin(_rms(self.lin(h, mix + "dq"), eps) * w[mix + "dq.norm"].double(), mix + "uq").view(n, heads, -1)
            q_rot = _rotate(q[..., dim:], at, base)
            keys, values = self.lin(latent, mix + "uk").view(n, heads, -1), self.lin(latent, mix + "uv").view(n, heads, -1)
            gates, out = self.lin(h, mix + "g").sigmoid(), []
            for a in range(heads):
                scores = (q[:, a, :dim] @ keys[:, a].t() + q_rot[:, a] @ k_rot.t()) * m["scale"]
                out.append(scores.masked_fill(~sees, -math.inf).softmax(1) @ values[:, a] * gates[:, a:a + 1])
            x = x + norm(self.lin(torch.cat(out, 1), mix + "o"), p + "norm1b")
            h = norm(x, p + "norm2")
            if f["kind"] == "dense":
                y = ff(h, mlp)
            else:
                chosen = w[mlp + "table"][ids].long()
                y = self.expert_sum(h, chosen, torch.full(chosen.shape, 1.0 / chosen.shape[1], dtype=torch.float64, device="cuda"),
                                    lambda r, e: ff(r, mlp + f"e{e}.")) + ff(h, mlp + "shared.")
            states.append(x + norm(y, p + "norm2b"))
            x = sum(a * s for a, s in zip(w[p + "dwa"].double(), states))
        return norm(x, "final.norm")

    def memory(self, h, m, mix, eps):
        n, heads, dim, vdim, cap = len(h), m["heads"], m["dim"], m["vdim"], m["gate_cap"]
        q, k = self.lin(h, mix + "q").view(n, heads, dim) * dim ** -0.5, self.lin(h, mix + "k").view(n, heads, dim)
        v = self.lin(h, mix + "v").view(n, heads, vdim)

        def capped(name):
            return cap * torch.tanh((self.lin(h, mix + name) + self.w[mix + name + ".b"].double()) / cap)

        log_in, kept = capped("i"), torch.nn.functional.logsigmoid(capped("f")).cumsum(0)
        causal = torch.ones(n, n, dtype=torch.bool, device="cuda").tril()
        out = []
        for a in range(heads):
            # entry (t, s): the log of what is left at t of what came in at s; the state starts at zero with scale 1
            left = (kept[:, a, None] - kept[None, :, a] + log_in[None, :, a]).masked_fill(~causal, -math.inf)
            top = torch.maximum(left.amax(1), kept[:, a])
            share = (left - top[:, None]).exp() * (q[:, a] @ k[:, a].t())
            out.append(share @ v[:, a] / (torch.maximum(share.sum(1).abs(), (-top).exp()) + 1e-6)[:, None])
        y = _rms(torch.stack(out, 1), eps).view(n, heads * vdim) * self.w[mix + "norm"].double() * self.lin(h, mix + "g").sigmoid()
        return self.lin(y, mix + "o")

    def attention(self, h, m, mix, at):
        n, heads, kv, dims = len(h), m["heads"], m["kv_heads"], m["rot"]["dims"]
        q, k = (self.lin(h, mix + name).view(n, -1, m["dim"]) for name in "qk")
        q, k = (torch.cat([_rotate(t[..., :dims], at, m["rot"]["base"]), t[..., dims:]], -1) for t in (q, k))
        v, sees, out = self.lin(h, mix + "v").view(n, kv, -1), _mask(at, at, m["mask"]["size"]), []
        for a in range(heads):
            scores = (q[:, a] @ k[:, a * kv // heads].t() * m["scale"]).masked_fill(~sees, -math.inf)
            sink = torch.cat([scores, torch.zeros(n, 1, dtype=torch.float64, device="cuda")], 1)
            out.append(sink.softmax(1)[:, :-1] @ v[:, a * kv // heads])
        return self.lin(torch.cat(out, 1), mix + "o")

    def dimesun(self, ids, at):
        cfg, w = self.cfg, self.w
        eps = cfg["norm"]["eps"]
        x = w["embed"][ids].double()
        for turn in range(cfg["loop"]["times"]):
            x = x + w["loop.step"][turn].double()
            for i, layer in enumerate(cfg["layers"]):
                p, m, f = f"l{i}.", layer["mixer"], layer["mlp"]
                mlp, limit = p + "mlp.", f["expert"]["limit"]
                h = _rms(x, eps) * (1.0 + w[p + "norm1"].double())
                y = self.memory(h, m, p + "mix.", eps) if layer["type"] == "mlstm" else self.attention(h, m, p + "mix.", at)
                logits = self.lin(h, mlp + "router") + w[mlp + "router.b"].double()
                best, chosen = logits.topk(f["router"]["top"], 1)

                def one(r, e):
                    gate = self.lin(r, mlp + f"e{e}.gate").clamp(max=limit)
                    return self.lin(gate * (1.702 * gate).sigmoid() * (self.lin(r, mlp + f"e{e}.up").clamp(-limit, limit) + 1.0),
                                    mlp + f"e{e}.down")

                x = x + cfg["residual_mult"] * (y + self.expert_sum(h, chosen, best.softmax(1), one))
        return _rms(x, eps) * (1.0 + w["final.norm"].double())


def exact(case, seed):
    if case["what"] in ("linear", "row"):
        g = _generator(seed)
        shapes = [("", case["out"], case["in"])] if case["what"] == "linear" else _row_shapes(case)
        weights = {name: _layer_weight(g, n, k) for name, n, k in shapes}
        if case["what"] == "linear":
            return _linear_exact(weights[""], _activations(g, case["rows"], case["in"]))
        x, attention = _activations(g, 1, case["hidden"]), _normal(g, 1, case["hidden"])
        h, act = _activations(g, 1, case["hidden"]), _normal(g, 1, case["ffn"])
        rows = {"q": x, "k": x, "v": x, "o": attention, "gate": h, "up": h, "down": act}
        return [_linear_exact(weights[name], rows[name]) for name, _, _ in shapes]
    ids, prompt, new = _tokens(case, seed), case["tokens"], case.get("new", 0)
    if case["model"] == "qwen3":
        model = _Qwen3Exact(case)
        if case["what"] == "prompt":
            return model.forward(ids)
        logits = [model.forward(ids[:prompt])]
        if case["what"] == "steps":
            return logits + [model.forward(ids[i:i + 1]) for i in range(prompt, len(ids))]
        tokens = [int(logits[0].argmax())]
        for _ in range(new - 1):
            tokens.append(int(model.forward(tokens[-1:]).argmax()))
        return np.array(tokens, np.int32), model.forward(tokens[-1:])
    model = _DenseExact(case)
    if case["what"] == "prompt":
        return model.forward(ids, 1)
    if case["what"] == "steps":
        return list(model.forward(ids, new + 1).split(1))
    tokens = ids[:prompt].tolist()
    for _ in range(new):
        tokens.append(int(model.forward(tokens, 1).argmax()))
    return np.array(tokens[prompt:], np.int32), model.forward(tokens, 1)
