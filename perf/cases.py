"""The work whose time counts: prompts, generation and served batches through the public entry points.

Every case is a model of this repository's own configurations (the LLaMA sizes, the two-layer plumbing model, the layered hybrid of the
benchmark) with random weights in the statistics of a checkpoint, and one thing a program does with it:

  generate   `generate(model, idx, new)`, then the logits of one more token through `model(idx, S, input_pos)`, then `reset_cache()`: a sample
             of generate.py, prompt included
  prompt     `model(idx, S, input_pos)` over a whole prompt, the logits of every position
  serve      a hybrid model's engine: packed prompts of a batch, a few decode steps, slots given back
  decode     a hybrid model's engine: decode steps of sequences whose prompts went in before

The head of a LLaMA is its embedding with the rows dealt out anew, so that one next token stands out by far, as in a trained model: greedy and
sampled tokens do not hang on a rounding.
"""
from __future__ import annotations

import functools
import math

import torch

from lit_llama_amd import generate
from lit_llama_amd.hybrid import HybridConfig, HybridLM
from lit_llama_amd.hybrid_engine import Entry
from lit_llama_amd.model import LLaMA, LLaMAConfig
from lit_llama_amd.quantization import ColBlockQuantizedLinear
from lit_llama_amd.utils import EmptyInitOnDevice

VOCAB = 32000
HEADS = {256: 4, 4096: 32, 5120: 40, 6656: 52, 8192: 64}  # heads by width: the plumbing model, 7B, 13B, 30B, 65B
CACHE = 4096  # positions a hybrid engine's caches are sized for
GLA_RANK = 16  # low rank of a gated linear attention's decay


def _llama(name, kind, fmt, width, layers, prompt, new=0, top_k=1):
    return {"name": name, "kind": kind, "fmt": fmt, "width": width, "layers": layers, "prompt": prompt, "new": new, "top_k": top_k}


def _hybrid(name, kind, width, layers, batch, prompt, steps):
    return {"name": name, "kind": kind, "fmt": "bf16", "width": width, "layers": layers, "batch": batch, "prompt": prompt, "steps": steps}


def listed():
    return [
        # the plumbing model: what a call costs when there is hardly anything to compute
        _llama("plumbing generate 6+6", "generate", "int4", 256, 2, 6, 6),
        # a chat turn of the headline model (7B gptq.int4, one sequence)
        _llama("7B int4 generate 128+64", "generate", "int4", 4096, 32, 128, 64),
        # a document as long as the context
        _llama("7B int4 prompt 2048", "prompt", "int4", 4096, 32, 2048),
        # a short question
        _llama("7B int4 prompt 37", "prompt", "int4", 4096, 32, 37),
        # GPTQ checkpoints with a group size of 128
        _llama("7B int4-g128 prompt 1000", "prompt", "int4-g128", 4096, 8, 1000),
        # the unquantised model, sampled as the command line does it
        _llama("7B bf16 sampled 24+32", "generate", "bf16", 4096, 32, 24, 32, 200),
        _llama("7B bf16 prompt 777", "prompt", "bf16", 4096, 8, 777),
        # LLM.int8, two layers: activations are rounded to 8 bits in front of every product, so that two correct programs whose sums
        # differ in the last bit are some per cent apart a few layers on (8 layers: 0.04 of the result's norm, 32 layers: 0.06)
        _llama("7B int8 generate 200+24", "generate", "int8", 4096, 2, 200, 24),
        _llama("7B int8 prompt 512", "prompt", "int8", 4096, 2, 512),
        # a larger model
        _llama("13B int4 generate 50+32", "generate", "int4", 5120, 40, 50, 32),
        # the hybrid family: one long prompt with its first tokens, and a batch that decodes
        _hybrid("hybrid serve 1 x 2048", "serve", 4096, 8, 1, 2048, 2),
        _hybrid("hybrid decode 16", "decode", 4096, 8, 16, 1536, 4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.3:
        batch = _log(rng, 1, 64)
        c = _hybrid("", rng.choice(["serve", "decode"]), rng.choice([2048, 3072, 4096, 5120]), rng.choice([4, 8]), batch,
                    _log(rng, 1, min(2048, 8192 // batch)), rng.randint(1, 6))
    else:
        width = rng.choice([256, 4096, 4096, 4096, 5120, 6656, 8192])
        layers = rng.randint(1, {256: 8, 4096: 12, 5120: 8, 6656: 5, 8192: 4}[width])
        fmt = rng.choice(["int4", "int4", "int4-g128", "bf16", "int8", "gptq8"])
        layers = min(layers, 2) if fmt == "int8" else layers
        if rng.random() < 0.5:
            c = _llama("", "prompt", fmt, width, layers, _log(rng, 2, 2048))
        else:
            c = _llama("", "generate", fmt, width, layers, _log(rng, 1, 1024), _log(rng, 2, 64), rng.choice([1, 200]))
    del c["name"]
    return c


# ---------------------------------------------------------------------------------------- weights
def _gen(seed, *path):
    s = seed
    for p in path:
        s = (s * 1000003 + p + 12345) % (2 ** 61 - 1)
    return torch.Generator(device="cuda").manual_seed(s)


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _hidden(width):
    return -(-int(8 * width / 3) // 256) * 256


def _config(case):
    return LLaMAConfig(n_layer=case["layers"], n_head=HEADS[case["width"]], n_embd=case["width"])


def _shapes(width):
    h = _hidden(width)
    return [("attn.c_attn", 3 * width, width), ("attn.c_proj", width, width), ("mlp.c_fc1", h, width), ("mlp.c_fc2", h, width), ("mlp.c_proj", width, h)]


def _grid(w, fmt):
    """Round to nearest on a grid per row, or per row and 128 columns: levels, scales, zeros (whole numbers)."""
    top = 255 if fmt == "gptq8" else 15
    x = w.view(w.shape[0], -1, 128 if fmt == "int4-g128" else w.shape[1])
    lo, hi = x.amin(2, keepdim=True).clamp(max=0), x.amax(2, keepdim=True).clamp(min=0)
    scale = ((hi - lo) / top).bfloat16().float()
    zero = torch.round(-lo / scale)
    return (torch.round(x / scale) + zero).clamp_(0, top), scale, zero


def _stored(w, fmt, name):
    """The checkpoint's tensors of a linear layer with the weights w."""
    if fmt in ("bf16", "int8"):
        return {name + ".weight": w.bfloat16()}
    q, scale, zero = _grid(w, fmt)
    q = q.view(w.shape).to(torch.uint8)
    if fmt != "gptq8":
        q = q[:, ::2] | (q[:, 1::2] << 4)
    return {name + ".quant_weight": q, name + ".scales": scale.squeeze(2).bfloat16(), name + ".zeros": zero.squeeze(2).bfloat16()}


def _llama_parts(case, seed):
    """(name, f32 weights) of every linear layer, then the other tensors, one at a time."""
    C, fmt = case["width"], case["fmt"]
    for i in range(case["layers"]):
        g = _gen(seed, 1, i)
        for name, n, k in _shapes(C):
            yield f"transformer.h.{i}.{name}", _randn(g, n, k) * k ** -0.5
        for j in (1, 2):
            yield f"transformer.h.{i}.rms_{j}.scale", (1 + 0.1 * _randn(g, C)).bfloat16()
    g = _gen(seed, 2)
    wte = _randn(g, VOCAB, C).bfloat16()
    head = torch.empty_like(wte, dtype=torch.float32)
    head[_next_of(seed)] = wte.float() * 3 * C ** -0.5
    yield "transformer.wte.weight", wte
    yield "transformer.ln_f.scale", (1 + 0.1 * _randn(g, C)).bfloat16()
    yield "lm_head", head


def _next_of(seed):
    return torch.randperm(VOCAB, generator=_gen(seed, 3), device="cuda")


def _prompt(seed, n, i=0):
    return torch.randint(0, VOCAB, (n,), generator=_gen(seed, 4, i), device="cuda", dtype=torch.int32)


def _hybrid_conf(case):
    """The benchmark's hybrid: window attention | gated linear attention | window attention | gated delta rule in turn."""
    width = case["width"]
    heads, ff = width // 128, _hidden(width) * 3 // 2
    att = {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5}
    mixers = [("attention", {**att, "rot": {"base": 1e4, "dims": 128}, "mask": {"size": 2048}}),
              ("gla", {"heads": heads, "dim": 128, "vdim": 128, "tau": 16.0}),
              ("attention", {**att, "rot": {"base": 1e4, "dims": 64}, "mask": {"size": 1024}}),
              ("delta", {"heads": heads, "kv_heads": heads // 2, "dim": 128, "vdim": 128, "conv": 4})]
    layers = [{"type": t, "mixer": m, "mlp": {"kind": "dense", "ff": ff}} for t, m in (mixers[i % 4] for i in range(case["layers"]))]
    return {"architecture": "Sekulorn", "layers": layers, "loop": None, "norm": {"eps": 1e-5}, "residual_mult": 1.0, "vocab": VOCAB, "width": width}


def _hybrid_layer(case, seed, i):
    """Tensors of layer i: unit-gain projections, decays around 0.9, so that far tokens still count."""
    W, g = case["width"], _gen(seed, 5, i)
    spec = _hybrid_conf(case)["layers"][i]
    m, ff = spec["mixer"], spec["mlp"]["ff"]
    hv, gk = m["heads"] * m["vdim"], m.get("kv_heads", m["heads"]) * m["dim"]
    lin = lambda n, k: (_randn(g, n, k) * k ** -0.5).bfloat16()  # noqa: E731
    vec = lambda n, scale, at: (at + scale * _randn(g, n)).bfloat16()  # noqa: E731

    def conv(n):
        t = 0.2 * _randn(g, n, m["conv"])
        t[:, -1] += 0.7
        return t.bfloat16()

    t = {"norm1": vec(W, 0.1, 1), "norm2": vec(W, 0.1, 1), "mlp.up": lin(ff, W), "mlp.down": lin(W, ff), "mix.o": lin(W, hv)}
    if spec["type"] == "attention":
        t.update({"mix.q": lin(m["heads"] * m["dim"], W), "mix.k": lin(gk, W), "mix.v": lin(m["kv_heads"] * m["vdim"], W), "mix.g": lin(m["heads"], W)})
    else:
        t.update({"mix.q": lin(gk, W), "mix.k": lin(gk, W), "mix.v": lin(hv, W), "mix.g": lin(hv, W), "mix.norm": vec(m["vdim"], 0.1, 1)})
    if spec["type"] == "gla":
        t.update({"mix.a1": lin(GLA_RANK, W), "mix.a2": lin(gk, GLA_RANK), "mix.a2.b": vec(gk, 0.5, 2)})
    if spec["type"] == "delta":
        t.update({"mix.q.conv": conv(gk), "mix.k.conv": conv(gk), "mix.v.conv": conv(hv), "mix.b": lin(m["heads"], W), "mix.a": lin(m["heads"], W),
                  "mix.A_log": vec(m["heads"], 0.3, -2), "mix.dt_bias": vec(m["heads"], 0.5, 0)})
    return t


def _hybrid_ends(case, seed):
    g = _gen(seed, 6)
    W = case["width"]
    return {"embed": _randn(g, VOCAB, W).bfloat16(), "final.norm": (1 + 0.1 * _randn(g, W)).bfloat16(),
            "head": (_randn(g, VOCAB, W) * W ** -0.5).bfloat16()}


def _lengths(case):
    """Prompts of a batch: from a part of the longest up to it."""
    return [-(-case["prompt"] * (i + 1) // case["batch"]) for i in range(case["batch"])]


def _sequences(case, seed):
    return [_prompt(seed, n + case["steps"], 1 + i) for i, n in enumerate(_lengths(case))]


# ---------------------------------------------------------------------------------------- the calls
def _build_llama(case, seed):
    fmt = case["fmt"]
    mode = {"int4": "gptq.int4", "int8": "llm.int8", "gptq8": "gptq.int8"}.get(fmt)
    with EmptyInitOnDevice(device="cuda", dtype=torch.bfloat16, quantization_mode=mode):
        dense = torch.nn.Linear
        if fmt == "int4-g128":
            torch.nn.Linear = functools.partial(ColBlockQuantizedLinear, bits=4, tile_cols=128)
        try:
            model = LLaMA(_config(case))
        finally:
            torch.nn.Linear = dense
    tensors = {}
    for name, w in _llama_parts(case, seed):
        tensors.update({name: w} if w.dtype == torch.bfloat16 else _stored(w, fmt, name))
    model.load_state_dict(tensors)
    model.eval()
    model.engine()
    return model


def prepare(case, seed):
    if case["kind"] in ("generate", "prompt"):
        n = case["prompt"]
        s = {"model": _build_llama(case, seed), "idx": _prompt(seed, n), "seed": seed, **{k: case[k] for k in ("kind", "new", "top_k")}}
        if case["kind"] == "prompt":
            s["pos"] = torch.arange(0, n, device="cuda")
        else:
            s["last"] = torch.tensor([n + case["new"] - 1], device="cuda")
        return s
    model = HybridLM(HybridConfig.from_dict(_hybrid_conf(case)), device="cuda")
    tensors = _hybrid_ends(case, seed)
    for i in range(case["layers"]):
        tensors.update({f"l{i}.{k}": v for k, v in _hybrid_layer(case, seed, i).items()})
    model.load_state_dict(tensors)
    eng = model.engine()
    eng.ensure(case["batch"], CACHE)
    s = {"model": model, "tokens": [t.tolist() for t in _sequences(case, seed)], "lengths": _lengths(case), "kind": case["kind"], "steps": case["steps"]}
    if case["kind"] == "decode":
        s["slots"] = [eng.acquire() for _ in s["lengths"]]
        eng.step([Entry(a, 0, t[:n], []) for a, t, n in zip(s["slots"], s["tokens"], s["lengths"])])
        s["done"] = 0
    return s


@torch.no_grad()
def run(state):
    if state["kind"] == "prompt":
        model, idx = state["model"], state["idx"]
        logits = model(idx.view(1, -1), idx.numel(), state["pos"])
        model.reset_cache()
        return {"logits": logits}
    if state["kind"] == "generate":
        model, idx = state["model"], state["idx"]
        torch.manual_seed(state["seed"])
        tokens = generate(model, idx, state["new"], temperature=0.8, top_k=state["top_k"])
        logits = model(tokens[-1:].view(1, 1), tokens.numel(), state["last"])
        model.reset_cache()
        return {"tokens": tokens, "logits": logits}
    eng, tokens, lengths, out = state["model"].engine(), state["tokens"], state["lengths"], []
    if state["kind"] == "serve":
        slots, done = [eng.acquire() for _ in lengths], 0
        out.append(eng.step([Entry(a, 0, t[:n], [n - 1]) for a, t, n in zip(slots, tokens, lengths)]).clone())
    else:  # the sequences go on from pass to pass, up to the end of their caches
        slots, done = state["slots"], state["done"]
        state["done"] = done + state["steps"] if max(lengths) + done + 2 * state["steps"] <= CACHE else 0
    for j in range(state["steps"]):
        out.append(eng.step([Entry(a, n + done + j, t[n + j:n + j + 1], [0]) for a, t, n in zip(slots, tokens, lengths)]).clone())
    if state["kind"] == "serve":
        for a in slots:
            eng.release(a)
    return {"logits": out}


# ---------------------------------------------------------------------------------------- what a pass cannot do without
def _weight_bytes(fmt):
    return {"int4": 0.5, "int4-g128": 0.5 + 4 / 128, "bf16": 2, "int8": 1, "gptq8": 1}[fmt]


def work(case):
    W, L = case["width"], case["layers"]
    if case["kind"] in ("generate", "prompt"):
        T, new = case["prompt"], case["new"]
        body, head = L * sum(n * k for _, n, k in _shapes(W)), VOCAB * W
        steps = new if case["kind"] == "generate" else 0  # behind the prompt: new - 1 tokens and the last logits
        rows = T if case["kind"] == "prompt" else 1       # whose logits the prompt gives
        seen = sum(range(T + 1, T + steps + 1))
        flops = 2 * body * (T + steps) + 2 * head * (rows + steps) + 2 * L * W * T * T + 4 * L * W * seen
        data = (body + head) * _weight_bytes(case["fmt"]) * (1 + steps) + 4 * L * W * (T + seen) + 4 * VOCAB * (rows if not steps else 1)
        return {"bytes": data, "flops": flops}
    B, steps, n = case["batch"], case["steps"], _lengths(case)
    body = state = 0
    for spec in _hybrid_conf(case)["layers"]:
        m, ff = spec["mixer"], spec["mlp"]["ff"]
        hv, gk = m["heads"] * m["vdim"], m.get("kv_heads", m["heads"]) * m["dim"]
        body += 2 * W * ff + W * hv + W * (hv + 2 * gk if spec["type"] == "attention" else 2 * gk + 2 * hv)
        if spec["type"] != "attention":
            state += 4 * m["heads"] * m["dim"] * m["vdim"]

    def attention(lo, hi):  # pairs of rows and keys over all attention layers, positions lo .. hi - 1
        return sum(sum(min(p + 1, s["mixer"]["mask"]["size"]) for p in range(lo, hi)) for s in _hybrid_conf(case)["layers"] if s["type"] == "attention")

    head, rows = VOCAB * W, B * steps
    flops, data = 2 * body * rows + 2 * head * rows, steps * 2 * (body + head) + 2 * B * steps * state + 4 * VOCAB * rows
    pairs = sum(attention(x, x + steps) for x in n)
    flops, data = flops + 4 * W * pairs, data + W * pairs  # (a quarter as many key heads, keys and values in bf16)
    if case["kind"] == "serve":
        flops += 2 * body * sum(n) + 2 * head * B + 4 * W * sum(attention(0, x) for x in n) + state * sum(n)
        data += 2 * (body + head) + B * state + 4 * VOCAB * B
    return {"bytes": data, "flops": flops}


def tolerance(case):
    """Measured against 64 bits: 0.004 to 0.0075 of the logits' norm over 2 to 40 layers with bf16 operands, 0.02 with LLM.int8 (rounding that
    goes the other way); four times the former.  Tokens stand out: none differs, but for one in a long run."""
    return {"rel": 0.03, "max": 0.3, "differ": 0.01}


# ---------------------------------------------------------------------------------------- the same in 64 bits
def _norm64(x, scale):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * scale


def _turn64(x, dims):
    """x [T, heads, dim], row t at position t: neighbours among the first `dims` dimensions turn by t * 10000^(-2i / dims)."""
    a = torch.arange(x.shape[0], device="cuda", dtype=torch.float64)[:, None] * 1e4 ** (-2.0 * torch.arange(dims // 2, device="cuda", dtype=torch.float64) / dims)
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    u, v = x[..., 0:dims:2], x[..., 1:dims:2]
    return torch.cat([torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2), x[..., dims:]], -1)


def _attend64(q, k, v, scale, window):
    """q [T, H, d], k and v [T, G, d]: row i sees the last `window` rows up to itself."""
    T, H, _ = q.shape
    i = torch.arange(T, device="cuda")
    far = i[:, None] - i[None, :]
    hide = (far < 0) | (far >= window)
    out = torch.empty_like(q)
    for h in range(H):
        g = h * k.shape[1] // H
        out[:, h] = torch.softmax((q[:, h] @ k[:, g].T * scale).masked_fill_(hide, -math.inf), -1) @ v[:, g]
    return out


def _eight64(x, w, first):
    """LLM.int8 of the rows x: those of a prompt (the first ones) share their outlier columns, later rows are calls of their own."""
    wh = w.bfloat16().half().double()
    scb = wh.abs().amax(1, keepdim=True)
    cb = torch.round(wh * (127 / scb))
    big = x.abs() >= 6
    sca = x.masked_fill(big, 0).abs().amax(1, keepdim=True)
    big[:first] = big[:first].any(0)
    ca = torch.round(x * (127 / sca)).masked_fill_(big, 0)
    return (ca * (sca / 127)) @ (cb * (scb / 127)).T + x.masked_fill(~big, 0) @ (cb * (scb / 127)).T


def _product64(x, w, fmt, first):
    if fmt == "int8":
        return _eight64(x, w, first)
    if fmt == "bf16":
        return x @ w.bfloat16().double().T
    q, scale, zero = _grid(w, fmt)
    return x @ ((q.double() - zero) * scale).view(w.shape).T


def _llama64(case, seed, tokens, rows):
    """Logits of the last `rows` positions."""
    C, H, fmt, first = case["width"], HEADS[case["width"]], case["fmt"], case["prompt"]
    parts, ends = _llama_parts(case, seed), {}
    layers = []
    x = _randn(_gen(seed, 2), VOCAB, C).bfloat16()[tokens.long()].double()
    hold = {}
    for name, w in parts:
        if not name.startswith("transformer.h."):
            ends[name] = w
            continue
        leaf = name.split(".", 3)[3]
        hold[leaf] = w
        if leaf != "rms_2.scale":
            continue
        T = x.shape[0]
        mul = lambda a, n: _product64(a, hold[n], fmt, first)  # noqa: E731
        q, k, v = mul(_norm64(x, hold["rms_1.scale"].double()), "attn.c_attn").view(T, 3, H, C // H).unbind(1)
        d = C // H
        x = x + mul(_attend64(_turn64(q, d), _turn64(k, d), v, d ** -0.5, T).reshape(T, C), "attn.c_proj")
        h = _norm64(x, hold["rms_2.scale"].double())
        x = x + mul(torch.nn.functional.silu(mul(h, "mlp.c_fc1")) * mul(h, "mlp.c_fc2"), "mlp.c_proj")
        hold = {}
    x = _norm64(x, ends["transformer.ln_f.scale"].double())
    first = max(0, first - (x.shape[0] - rows))
    if rows < x.shape[0] or case["kind"] == "generate":
        first = 1  # (each of these rows is a call of its own)
    return _product64(x[-rows:], ends["lm_head"], fmt, first)


def _conv64(x, taps):
    n = taps.shape[1]
    x = torch.nn.functional.pad(x, (0, 0, n - 1, 0))
    return sum(x[:, j:x.shape[1] - n + 1 + j] * taps[:, j] for j in range(n))


def _mix64(spec, w, h):
    """One mixer over h [B, T, width]."""
    m, (B, T, _) = spec["mixer"], h.shape
    H, G, d = m["heads"], m.get("kv_heads", m["heads"]), m["dim"]
    lin = lambda n: h @ w["mix." + n].T  # noqa: E731
    if spec["type"] == "attention":
        q, k, v = (lin(n).view(B, T, -1, d) for n in "qkv")
        dims = m["rot"]["dims"]
        o = torch.stack([_attend64(_turn64(q[b], dims), _turn64(k[b], dims), v[b], m["scale"], m["mask"]["size"]) for b in range(B)])
        return (o * torch.sigmoid(lin("g"))[..., None]).reshape(B, T, -1) @ w["mix.o"].T
    if spec["type"] == "gla":
        q, k, v = lin("q").view(B, T, H, d) * d ** -0.5, lin("k").view(B, T, H, d), lin("v").view(B, T, H, -1)
        keep = torch.sigmoid((lin("a1") @ w["mix.a2"].T + w["mix.a2.b"])).pow(1 / m["tau"]).view(B, T, H, d)
    else:
        q, k, v = (torch.nn.functional.silu(_conv64(lin(n), w[f"mix.{n}.conv"])) for n in "qkv")
        unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        q, k = (unit(t.view(B, T, G, d)).repeat_interleave(H // G, 2) for t in (q, k))
        q, v = q * d ** -0.5, v.view(B, T, H, -1)
        beta = torch.sigmoid(lin("b"))
        keep = torch.exp(-torch.exp(w["mix.A_log"]) * torch.nn.functional.softplus(lin("a") + w["mix.dt_bias"]))[..., None].expand(B, T, H, d)
    S, out = h.new_zeros(B, H, d, v.shape[-1]), torch.empty_like(v)
    for t in range(T):
        S = S * keep[:, t, :, :, None]
        u = v[:, t]
        if spec["type"] == "delta":
            u = beta[:, t, :, None] * (u - (k[:, t, :, None] @ S).squeeze(2))
        S = torch.addcmul(S, k[:, t, :, :, None], u[:, :, None])
        out[:, t] = (q[:, t, :, None] @ S).squeeze(2)
    return (_norm64(out, w["mix.norm"]).reshape(B, T, -1) * torch.nn.functional.silu(lin("g"))) @ w["mix.o"].T


def exact(case, seed):
    with torch.no_grad():
        if case["kind"] == "prompt":
            return {"logits": _llama64(case, seed, _prompt(seed, case["prompt"]), case["prompt"])[None]}
        if case["kind"] == "generate":
            follow, tokens = _next_of(seed), _prompt(seed, case["prompt"])
            for _ in range(case["new"]):
                tokens = torch.cat([tokens, follow[tokens[-1:].long()].int()])
            logits = _llama64(case, seed, tokens, case["new"] + 1)
            if not torch.equal(logits[:-1].argmax(-1).int(), tokens[case["prompt"]:]):
                raise AssertionError("the next token does not stand out")
            return {"tokens": tokens, "logits": logits[-1:][None]}
        seqs = _sequences(case, seed)
        if sum(t.numel() for t in seqs) * case["width"] ** 2 * case["layers"] > 5e12:
            return None
        T = max(t.numel() for t in seqs)
        ids = torch.stack([torch.nn.functional.pad(t, (0, T - t.numel())) for t in seqs]).long()
        ends = _hybrid_ends(case, seed)
        x = ends["embed"][ids].double()
        for i, spec in enumerate(_hybrid_conf(case)["layers"]):
            w = {k: v.double() for k, v in _hybrid_layer(case, seed, i).items()}
            x = x + _mix64(spec, w, _norm64(x, w["norm1"]))
            for b in range(x.shape[0]):
                x[b] += torch.relu(_norm64(x[b], w["norm2"]) @ w["mlp.up"].T).square() @ w["mlp.down"].T
        first = -1 if case["kind"] == "serve" else 0
        head = ends["head"].double().T
        final = ends["final.norm"].double()
        return {"logits": [torch.stack([_norm64(x[b, n + j], final) for b, n in enumerate(_lengths(case))]) @ head for j in range(first, case["steps"])]}
