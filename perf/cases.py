"""What is measured: passes of the inference engine on models of every family, each pass the whole life of a batch of requests.

A pass feeds B prompts of P tokens to Engine.feed (prefill), then S times the next token of every request (decode: the captured step
graph that generation replays), takes the logits behind each request's last token and ends the requests. Tokens are given, so that the
logits can be checked against 64 bits; generation runs the same step functions. Models have the layer shapes of the package's benchmark
(bench_stack.SIZES: widths 2048 and 4096, four layer runs, 32 000 words): the GGUF families with quantised weights, the config-driven
designs in bf16 or, with the `float32` option, in 32 bits throughout.

`exact` is each model in plain torch in 64 bits, with the weights made here."""
from __future__ import annotations

import functools
import json
import math
import os
import shutil
import tempfile

import numpy as np
import torch

from nats_llm_studio_amd import bench_stack
from nats_llm_studio_amd.engine.engine import Engine
from nats_llm_studio_amd.gguf.constants import FILE_TYPE_IDS, GGMLType
from nats_llm_studio_amd.gguf.writer import GGUFWriter
from nats_llm_studio_amd.models.registry import load_model
from nats_llm_studio_amd.safetensors_io import write_safetensors

VOCAB = bench_stack.VOCAB
DEVICE = torch.device("cuda:0")
BLOCK = 16
STACKS = ("sekolorn", "kolodra", "bibapel", "pimodra")
# GGUF shapes: width, heads, key heads, feed-forward, experts
GGUF = {
    ("llama", "2k"): dict(d=2048, H=16, G=4, ff=8192, E=0),
    ("llama", "4k"): dict(d=4096, H=32, G=8, ff=14336, E=0),
    ("mixtral", "2k"): dict(d=2048, H=16, G=4, ff=4096, E=8),
    ("mixtral", "4k"): dict(d=4096, H=32, G=8, ff=4096, E=8),
}
LAYERS, EPS, ROPE, TOP = 4, 1e-5, 500000.0, 2


def listed():
    def c(name, model, size, form, batch, prompt, steps):
        return dict(name=name, model=model, size=size, form=form, batch=batch, prompt=prompt, steps=steps)
    return [
        # one user's short question and its answer: the smallest launches, latency counts
        c("chat-1", "llama", "4k", "Q4_K_M", 1, 21, 32),
        # a loaded server, many short requests at once: the headline benchmark's kind of step
        c("batch-300", "llama", "4k", "Q4_K_M", 300, 20, 40),
        # a long document as prompt
        c("document-3000", "llama", "4k", "Q4_K_M", 1, 3000, 0),
        # routed experts of a GGUF file under a few dozen users
        c("experts-24", "mixtral", "2k", "Q5_K_M", 24, 90, 24),
        # each design's decoding under load, from a few users to a full batch
        c("kolodra-64", "kolodra", "4k", "bf16", 64, 60, 32),
        c("sekolorn-200", "sekolorn", "4k", "bf16", 200, 16, 24),
        c("bibapel-16", "bibapel", "4k", "bf16", 16, 130, 32),
        # and prompts: one long, several, a ragged burst of short ones behind few decoded tokens
        c("kolodra-prompt", "kolodra", "4k", "bf16", 1, 2000, 0),
        c("bibapel-prompts", "bibapel", "2k", "bf16", 6, 650, 0),
        c("sekolorn-prompt", "sekolorn", "2k", "bf16", 1, 3500, 0),
        c("pimodra-chats", "pimodra", "4k", "bf16", 9, 333, 6),
        # 32 bits throughout, as a reference run asks for
        c("kolodra-float32", "kolodra", "2k", "float32", 3, 300, 6),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    model = rng.choice(("llama", "llama", "mixtral") + STACKS)
    size = rng.choice(("2k", "4k"))
    if model in STACKS:
        form = rng.choice(("bf16", "bf16", "bf16", "float32"))
    else:
        form = rng.choice(("Q4_K_M", "Q4_K_M", "Q5_K_M", "Q8_0"))
    cap = 1500 if form == "float32" else 8000            # tokens of a pass
    if rng.random() < 0.5:                               # prompts
        prompt, steps = _log(rng, 16, 3500), rng.choice((0, 0, 3))
        batch = _log(rng, 1, 8)
    else:                                                # users
        batch, prompt, steps = _log(rng, 1, 300), _log(rng, 8, 300), rng.randint(8, 40)
    prompt = min(prompt, cap)
    steps = min(steps, 12) if form == "float32" else steps
    batch = max(1, min(batch, cap // prompt))
    return dict(model=model, size=size, form=form, batch=batch, prompt=prompt, steps=steps)


# ---- weights, made here

def _gen(text):
    return torch.Generator(device=DEVICE).manual_seed(sum(ord(ch) * 131 ** (i % 7) for i, ch in enumerate(text)) % (1 << 31))


def _k_scales(sc):
    """The 12 bytes of a K block's eight 6-bit scales, each also the sub-block's minimum."""
    lo, hi = sc[:, :4], sc[:, 4:]
    first = lo | (hi >> 4 << 6)
    return torch.cat([first, first, (hi & 15) | ((hi & 15) << 4)], 1)


def _half(n, v):
    return torch.full((n, 1), v, dtype=torch.float16, device=DEVICE).view(torch.uint8).view(n, 2)


def _blocks(kind, n, std, g):
    """n values as random blocks of a GGUF type, of zero mean and standard deviation std: bytes [blocks, bytes]."""
    def rand(rows, cols, lo=0, hi=256):
        return torch.randint(lo, hi, (rows, cols), generator=g, device=DEVICE, dtype=torch.uint8)
    if kind == "Q8_0":
        b = n // 32
        return torch.cat([_half(b, std / 73.6), rand(b, 32)], 1)
    b = n // 256
    if kind == "Q6_K":
        return torch.cat([rand(b, 192), rand(b, 16, 20, 44), _half(b, std / (32.5 * 18.5))], 1)
    top = {"Q4_K": 15, "Q5_K": 31}[kind]
    d = std / (32.5 * math.sqrt(((top + 1) ** 2 - 1) / 12))
    head = torch.cat([_half(b, d), _half(b, d * top / 2), _k_scales(rand(b, 8, 20, 44))], 1)
    return torch.cat([head, rand(b, 128 if kind == "Q4_K" else 160)], 1)


def _halves(x):
    return x.contiguous().view(torch.float16).double()


def _values(kind, raw):
    """The values of GGUF blocks, 64 bits."""
    n = raw.shape[0]
    if kind == "Q8_0":
        return (_halves(raw[:, :2]) * raw[:, 2:].contiguous().view(torch.int8).double()).reshape(-1)
    if kind == "Q6_K":
        ql, qh = raw[:, :128].view(n, 2, 64), raw[:, 128:192].view(n, 2, 32)
        a, b = ql[:, :, :32], ql[:, :, 32:]
        q = torch.stack([(a & 15) | ((qh & 3) << 4), (b & 15) | ((qh >> 2 & 3) << 4),
                         (a >> 4) | ((qh >> 4 & 3) << 4), (b >> 4) | ((qh >> 6) << 4)], 2)
        q = q.reshape(n, 16, 16).double() - 32
        sc = raw[:, 192:208].contiguous().view(torch.int8).double()
        return (_halves(raw[:, 208:])[:, :, None] * sc[:, :, None] * q).reshape(-1)
    d, dmin, s = _halves(raw[:, :2]), _halves(raw[:, 2:4]), raw[:, 4:16]
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6 << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6 << 4)], 1).double()
    qs = raw[:, -128:].view(n, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], 2).reshape(n, 8, 32)
    if kind == "Q5_K":
        bit = torch.arange(8, device=raw.device, dtype=torch.uint8)[None, :, None]
        q = q | ((raw[:, 16:48].view(n, 1, 32) >> bit & 1) << 4)
    return (d[:, :, None] * sc[:, :, None] * q.double() - dmin[:, :, None] * mn[:, :, None]).reshape(-1)


def _gguf_plan(model, size, form):
    """name -> (shape, GGUF type or None for 32-bit floats, mean, deviation)"""
    z = GGUF[model, size]
    base = form.replace("_M", "")
    more = "Q6_K" if form.endswith("_M") else base       # the recipe's bits of later values and down projections
    d, D, ff = z["d"], z["d"] // z["H"], z["ff"]
    plan = {"token_embd.weight": ((VOCAB, d), "Q8_0" if z["E"] else base, 0.0, 1.0)}
    for i in range(LAYERS):
        p, hi = f"blk.{i}.", more if i >= 2 else base
        ex = (z["E"],) if z["E"] else ()
        s = "_exps.weight" if z["E"] else ".weight"
        plan.update({p + "attn_norm.weight": ((d,), None, 1.0, 0.1), p + "ffn_norm.weight": ((d,), None, 1.0, 0.1),
                     p + "attn_q.weight": ((d, d), base, 0.0, d ** -0.5), p + "attn_k.weight": ((z["G"] * D, d), base, 0.0, d ** -0.5),
                     p + "attn_v.weight": ((z["G"] * D, d), hi, 0.0, d ** -0.5),
                     p + "attn_output.weight": ((d, d), base, 0.0, d ** -0.5),
                     p + "ffn_gate" + s: (ex + (ff, d), base, 0.0, d ** -0.5), p + "ffn_up" + s: (ex + (ff, d), base, 0.0, d ** -0.5),
                     p + "ffn_down" + s: (ex + (d, ff), hi, 0.0, ff ** -0.5)})
        if z["E"]:
            plan[p + "ffn_gate_inp.weight"] = ((z["E"], d), None, 0.0, d ** -0.5)
    plan.update({"output_norm.weight": ((d,), None, 1.0, 0.1), "output.weight": ((VOCAB, d), more, 0.0, d ** -0.5)})
    return plan


def _normal(name, mean, std, shape):
    return mean + std * torch.randn(shape, generator=_gen(name), device=DEVICE)


def _embedding(name, std, shape, routers):
    """Rows that lean towards two experts of every layer, as behind a trained router: a choice that hangs on a rounding is rare."""
    x, g = _normal(name, 0.0, std, shape), _gen(name + " experts")
    for r in routers:
        for e in torch.rand(shape[0], r.shape[0], generator=g, device=DEVICE).topk(TOP).indices.T:
            x += 10 * std * r[e]
    return x


def _gguf_tensor(plan, name):
    """A tensor as the file holds it: floats, or bytes [blocks, bytes]."""
    shape, kind, mean, std = plan[name]
    routers = [k for k in plan if "gate_inp" in k]
    if name == "token_embd.weight" and routers:
        x = _embedding(name, std, shape, [_gguf_tensor(plan, k) for k in routers]).view(-1, 32)
        d = (x.abs().amax(1, keepdim=True) / 127).half()
        return torch.cat([d.view(torch.uint8).view(-1, 2), torch.round(x / d.float()).clamp(-127, 127).to(torch.int8).view(torch.uint8)], 1)
    return _normal(name, mean, std, shape) if kind is None else _blocks(kind, math.prod(shape), std, _gen(name))


def _stack_plan(cfg):
    """name -> (mean, deviation, shape) of a design's checkpoint"""
    plan, d = {}, cfg["width"]
    arch = cfg["architecture"]
    # a sublayer whose output is normed adds less than the residual holds: that norm's weights are small
    small, scale = {"Sekolorn": (("norm1", "norm2"), 1.0), "Pimodra": (("norm1b", "norm2b"), 0.25)}.get(arch, ((), 1.0))

    def lin(name, *shape):
        plan[name] = 0.0, shape[-1] ** -0.5, shape

    def full(name, v, *shape):
        k = 0.4 * scale if name.count(".") == 1 and name.split(".")[1] in small else 1.0
        plan[name] = v * k, 0.1 * k, shape
    layer = getattr(bench_stack, f"_{arch.lower()}_layer")       # (the list of a layer's tensors)
    for i, L in enumerate(cfg["layers"]):
        layer(f"l{i}.", L, d, lin, full, *([cfg["rank"]] if "rank" in cfg else []))
    plan["embed"] = 0.0, d ** -0.5 if arch == "Bibapel" else scale, (VOCAB, d)
    full("final.norm", 0.0 if arch == "Kolodra" else 1.0, d)
    if arch == "Bibapel":
        plan["bigram"] = 0.0, d ** -0.5, (cfg["embedding"]["bigram"]["buckets"] + 1, d)
        plan["pos"] = 0.0, d ** -0.5, (cfg["max_positions"], d)
        lin("loop.in", d, 2 * d)
    if cfg.get("loop"):
        lin("loop.step", cfg["loop"]["times"], d)
    if arch in ("Sekolorn", "Kolodra"):
        lin("head", VOCAB, d)
    return plan


def _stack_tensor(plan, name):
    mean, std, shape = plan[name]
    if name == "embed":
        x = _embedding(name, std, shape, [_stack_tensor(plan, k).float() for k in plan if k.endswith("mlp.router")])
    else:
        x = _normal(name, mean, std, shape)
    return x.to(torch.bfloat16)


def _config(model, size):
    return bench_stack.CONFIGS[model](bench_stack.SIZES[model][size])


# ---- models and engines, loaded once as a worker keeps them

@functools.lru_cache(maxsize=24)
def _model(model, size, form):
    folder = tempfile.mkdtemp()
    try:
        if model in STACKS:
            cfg = _config(model, size)
            plan = _stack_plan(cfg)
            write_safetensors(os.path.join(folder, "model.safetensors"), {k: _stack_tensor(plan, k) for k in plan})
            with open(os.path.join(folder, "config.json"), "w") as f:
                json.dump({k: v for k, v in cfg.items() if k != "rank"}, f)
            return load_model(folder, DEVICE, dtype=torch.float32 if form == "float32" else torch.bfloat16, ctx=8192)
        z, path = GGUF[model, size], os.path.join(folder, "model.gguf")
        w = GGUFWriter(path, "llama")
        for k, v in {"general.name": model, "general.file_type": FILE_TYPE_IDS[form], "llama.context_length": 8192,
                     "llama.embedding_length": z["d"], "llama.block_count": LAYERS, "llama.feed_forward_length": z["ff"],
                     "llama.attention.head_count": z["H"], "llama.attention.head_count_kv": z["G"],
                     "llama.rope.freq_base": ROPE, "llama.rope.dimension_count": z["d"] // z["H"],
                     "llama.attention.layer_norm_rms_epsilon": EPS, "llama.vocab_size": VOCAB}.items():
            w.add(k, v)
        if z["E"]:
            w.add("llama.expert_count", z["E"])
            w.add("llama.expert_used_count", TOP)
        plan = _gguf_plan(model, size, form)
        for name, (shape, kind, _, _) in plan.items():
            w.add_tensor(name, shape, GGMLType[kind or "F32"],
                         lambda name=name: _gguf_tensor(plan, name).cpu().numpy().reshape(-1).view(np.uint8))
        w.write(None)
        return load_model(path, DEVICE)
    finally:
        shutil.rmtree(folder)


@functools.lru_cache(maxsize=24)
def _engine(model, size, form, batch, prompt, steps):
    tokens = prompt + steps
    eng = Engine(_model(model, size, form), None, max_batch=64 if batch <= 64 else 512, block_size=BLOCK,
                 num_blocks=batch * -(-tokens // BLOCK) + 8, max_prefill_tokens=4096, ctx=-(-tokens // BLOCK) * BLOCK + BLOCK,
                 prefix_cache=False)
    warm = torch.zeros(batch, tokens, dtype=torch.int64).tolist()
    for _ in range(2):                                    # a worker's warm-up: step graphs, scratch
        run(dict(engine=eng, ids=warm, prompt=prompt))
    return eng


def _ids(case, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, VOCAB, (case["batch"], case["prompt"] + case["steps"]), generator=g)


def prepare(case, seed):
    """The loaded engine and the requests' tokens."""
    eng = _engine(*(case[k] for k in ("model", "size", "form", "batch", "prompt", "steps")))
    return dict(engine=eng, ids=_ids(case, seed).tolist(), prompt=case["prompt"])


def run(state):
    """Logits [batch, words] behind the last token of each request."""
    eng, ids, P = state["engine"], state["ids"], state["prompt"]
    n = len(ids[0])
    out = eng.feed([(r, t[:P], [P - 1] if n == P else []) for r, t in enumerate(ids)])
    for k in range(P, n):
        out = eng.feed([(r, [t[k]], [0] if k == n - 1 else []) for r, t in enumerate(ids)])
    for r in range(len(ids)):
        eng.feed_end(r)
    return torch.cat(out)


# ---- what a pass cannot do without

def _sizes(case):
    """Bytes of the weights, (weights a token's products use, bytes of the experts, experts, top), cache bytes and attention operations
    per pair of a token and a key, state bytes."""
    z = GGUF.get((case["model"], case["size"]))
    dense = nbytes = eb = 0
    if z:
        for name, (shape, kind, _, _) in _gguf_plan(case["model"], case["size"], case["form"]).items():
            n = math.prod(shape)
            b = n * {"Q4_K": 144 / 256, "Q5_K": 176 / 256, "Q6_K": 210 / 256, "Q8_0": 34 / 32, None: 4}[kind]
            if name == "token_embd.weight":
                continue
            if "_exps" in name:
                eb, dense = eb + b, dense + n * TOP / z["E"]
            else:
                nbytes, dense = nbytes + b, dense + n
        return nbytes, dense, eb, z["E"], TOP, LAYERS * 4 * z["d"] // z["H"] * z["G"], LAYERS * 4 * z["d"], 0
    cfg = _config(case["model"], case["size"])
    el = 4 if case["form"] == "float32" else 2
    tied = case["model"] in ("bibapel", "pimodra")
    loop = cfg.get("loop") or {"start": 0, "stop": 0, "times": 1}
    runs = [loop["times"] if loop["start"] <= i < loop["stop"] else 1 for i in range(len(cfg["layers"]))]
    E = top = kv = pair = state = 0
    for name, (_, _, shape) in _stack_plan(cfg).items():
        if name in ("bigram", "pos") or (name == "embed" and not tied):
            continue
        n = math.prod(shape)
        layer = int(name[1:name.index(".")]) if name[0] == "l" and name[1].isdigit() else None
        r = 1 if layer is None else runs[layer]
        if ".mlp.e" in name:
            router = cfg["layers"][layer]["mlp"]["router"]
            E, top = router["experts"], router["top"]
            eb, dense = eb + r * n * el, dense + r * n * top / E
        else:
            nbytes, dense = nbytes + r * n * el, dense + (r * n if len(shape) > 1 else 0)
    for L, r in zip(cfg["layers"], runs):
        for m in ([L["mixer"]["left"], L["mixer"]["right"]] if L["type"] == "parallel" else [L["mixer"]]):
            if "kv_rank" in m:
                kv += r * el * (m["kv_rank"] + m["rot_dim"]) * ("kv_from" not in m)
                pair += r * 2 * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
            elif "scale" in m:
                kv += r * el * m["kv_heads"] * (m["dim"] + m["vdim"])
                pair += r * 2 * m["heads"] * (m["dim"] + m["vdim"])
            else:
                state += r * 8 * m["heads"] * m["dim"] * m.get("vdim", m["dim"])
    return nbytes, dense, eb, E, top, kv, pair, state


def work(case):
    nbytes, dense, eb, E, top, kv, pair, state = _sizes(case)
    B, P, S = case["batch"], case["prompt"], case["steps"]
    n = P + S
    head = VOCAB * (4096 if case["size"] == "4k" else 2048)
    out = nbytes + eb * (min(1.0, B * P * top / E) if E else 0)
    step = nbytes + eb * (min(1.0, B * top / E) if E else 0) + B * state + B * kv * (P + S / 2)
    return {"bytes": out + S * step + B * VOCAB * 4,
            "flops": 2 * (dense - head) * B * n + 2 * head * B * (1 + S) + pair * B * n * n / 2}


def tolerance(case):
    """About four times the distance from 64 bits that rounding leaves: f16 activations over quantised weights (0.002), bf16
    activations (0.007), 32-bit sums (2e-6)."""
    return {"rel": 1e-5 if case["form"] == "float32" else 0.03 if case["form"] == "bf16" else 0.01}


# ---- the models in 64 bits

class _Lazy:
    """name -> 64-bit tensor, made when asked for."""

    def __init__(self, fn):
        self.fn = fn

    def __getitem__(self, name):
        return self.fn(name)


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _rope(x, base, dims, gain=1.0, freq=None, halves=False):
    """Rotation of the first dims columns of x [B, n, heads, D] by position: neighbours, or one half with the other, are pairs."""
    f = torch.tensor(freq if freq is not None else [base ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=x.dtype, device=x.device)
    a = torch.arange(x.shape[1], dtype=x.dtype, device=x.device)[:, None, None] * f
    c, s = torch.cos(a) * gain, torch.sin(a) * gain
    h = dims // 2
    u, v = (x[..., :h], x[..., h:dims]) if halves else (x[..., 0:dims:2], x[..., 1:dims:2])
    u, v = u * c - v * s, v * c + u * s
    y = torch.cat([u, v], -1) if halves else torch.stack([u, v], -1).flatten(-2)
    return torch.cat([y, x[..., dims:]], -1)


def _attend(q, k, v, scale, window=0, keep=0, sink=False, talk=None):
    """q [B, n, H, D], k and v [B, n, G, ..]: causal attention, in parts of the batch and the rows that fit the card."""
    B, n, H, _ = q.shape
    r = H // k.shape[2]
    k, v = k.repeat_interleave(r, 2).permute(0, 2, 3, 1), v.repeat_interleave(r, 2).permute(0, 2, 1, 3)
    out = torch.empty(B, n, H, v.shape[-1], dtype=q.dtype, device=q.device)
    j = torch.arange(n, device=q.device)
    rows = max(1, min(n, (1 << 27) // (H * n)))
    seqs = max(1, (1 << 27) // (H * n * rows))
    for b in range(0, B, seqs):
        for i in range(0, n, rows):
            at = j[i:i + rows, None]
            see = j <= at
            if window:
                see = see & ((at - j < window) | (j < keep))
            s = (q[b:b + seqs, i:i + rows].transpose(1, 2) @ k[b:b + seqs] * scale).masked_fill(~see, -math.inf)
            if sink:
                m = s.amax(-1, keepdim=True).clamp(min=0.0)
                e = torch.exp(s - m)
                w = e / (torch.exp(-m) + e.sum(-1, keepdim=True))
            else:
                w = torch.softmax(s, -1)
            if talk is not None:
                w = (talk @ w.flatten(2)).view(w.shape)
            out[b:b + seqs, i:i + rows] = (w @ v[b:b + seqs]).transpose(1, 2)
    return out


def _experts(h, chosen, weight, expert):
    """Sum over a token's chosen experts; h [B, n, d], chosen and weight [B, n, top]."""
    x, c, w = h.flatten(0, 1), chosen.flatten(0, 1), weight.flatten(0, 1)
    out = torch.zeros_like(x)
    for e in range(int(c.max()) + 1):
        row, at = (c == e).nonzero(as_tuple=True)
        if len(row):
            out.index_add_(0, row, expert(e, x[row]) * w[row, at][:, None])
    return out.view(h.shape)


def _scan(n, S, step):
    out = []
    for t in range(n):
        o, S = step(t, S)
        out.append(o)
    return torch.stack(out, 1)


def _decayed(q, k, v, a):
    """The state S[key, value] decays by a, takes k v and is read by q; all [B, n, heads, ..]."""
    def step(t, S):
        S = a(t)[..., None] * S + k[:, t, :, :, None] * v[:, t, :, None, :]
        return (q[:, t, :, None, :] @ S)[..., 0, :], S
    return _scan(q.shape[1], torch.zeros(*q.shape[:1], *q.shape[2:], v.shape[-1], dtype=q.dtype, device=q.device), step)


def _llama(case, ids):
    plan = _gguf_plan(case["model"], case["size"], case["form"])
    z = GGUF[case["model"], case["size"]]
    H, G, D = z["H"], z["G"], z["d"] // z["H"]

    def get(name):
        shape, kind = plan[name][:2]
        t = _gguf_tensor(plan, name)
        return (t.double() if kind is None else _values(kind, t)).view(shape)
    W, (B, n) = _Lazy(get), ids.shape
    x = W["token_embd.weight"][ids]
    for i in range(LAYERS):
        p = f"blk.{i}."
        h = _rms(x, EPS) * W[p + "attn_norm.weight"]
        q, k, v = ((h @ W[p + f"attn_{s}.weight"].T).view(B, n, -1, D) for s in "qkv")
        o = _attend(_rope(q, ROPE, D), _rope(k, ROPE, D), v, D ** -0.5)
        x = x + o.flatten(2) @ W[p + "attn_output.weight"].T
        h = _rms(x, EPS) * W[p + "ffn_norm.weight"]
        if z["E"]:
            s, c = torch.softmax(h @ W[p + "ffn_gate_inp.weight"].T, -1).topk(TOP, -1)
            g, u, dn = (W[p + f"ffn_{s_}_exps.weight"] for s_ in ("gate", "up", "down"))
            x = x + _experts(h, c, s / s.sum(-1, keepdim=True), lambda e, r: (_silu(r @ g[e].T) * (r @ u[e].T)) @ dn[e].T)
        else:
            x = x + (_silu(h @ W[p + "ffn_gate.weight"].T) * (h @ W[p + "ffn_up.weight"].T)) @ W[p + "ffn_down.weight"].T
    return (_rms(x[:, -1], EPS) * W["output_norm.weight"]) @ W["output.weight"].T


def _layer_norm(x, w, eps):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _shares(s, router, best):
    """The chosen experts of score rows s, of the kept groups."""
    g = router.get("groups") or {"count": 1, "keep": 1}
    per = s.view(*s.shape[:-1], g["count"], -1)
    score = per.topk(min(best, per.shape[-1]), -1).values.sum(-1)
    kept = torch.zeros_like(score).scatter(-1, score.topk(g["keep"], -1).indices, 1.0)
    c = (per + 10.0 * kept[..., None]).flatten(-2).topk(router["top"], -1).indices
    return c, s.gather(-1, c)


def _sekolorn(cfg, W, ids):
    eps, (B, n) = cfg["norm"]["eps"], ids.shape
    x, rows = W["embed"][ids], {}
    for i, L in enumerate(cfg["layers"]):
        m, p = L["mixer"], f"l{i}.mix."
        if L["type"] == "wkv":
            sh = (B, n, m["heads"], m["dim"])
            back = torch.cat([torch.zeros_like(x[:, :1]), x[:, :-1]], 1) - x
            mix = {s: x + back * W[p + "mu." + s] for s in "rkvgw"}
            r, k, v = ((mix[s] @ W[p + s].T).view(sh) for s in "rkv")
            w = torch.exp(-torch.exp(torch.tanh(mix["w"] @ W[p + "w1"].T) @ W[p + "w2"].T + W[p + "w0"])).view(sh)
            u = W[p + "u"]

            def step(t, S):
                kv = k[:, t, :, :, None] * v[:, t, :, None, :]
                return (r[:, t, :, None, :] @ (S + u[:, :, None] * kv))[..., 0, :], w[:, t, :, :, None] * S + kv
            o = _scan(n, torch.zeros(B, *sh[2:], m["dim"], dtype=x.dtype, device=x.device), step)
            y = (_rms(o, eps).flatten(2) * W[p + "norm"] * _silu(mix["g"] @ W[p + "g"].T)) @ W[p + "o"].T
        else:
            H, D, R, RD = m["heads"], m["dim"], m["kv_rank"], m["rot_dim"]
            if "kv_from" not in m:
                c = x @ W[p + "dkv"].T
                rows[i] = _rms(c[..., :R], eps) * W[p + "dkv.norm"], _rope(c[:, :, None, R:], m["rot"]["base"], RD)
            c, kr = rows[m.get("kv_from", i)]
            q = ((_rms(x @ W[p + "dq"].T, eps) * W[p + "dq.norm"]) @ W[p + "uq"].T).view(B, n, H, D + RD)
            q = torch.cat([q[..., :D], _rope(q[..., D:], m["rot"]["base"], RD)], -1)
            k = torch.cat([(c @ W[p + "uk"].T).view(B, n, H, D), kr.expand(B, n, H, RD)], -1)
            o = _attend(q, k, (c @ W[p + "uv"].T).view(B, n, H, -1), m["scale"])
            y = (o * torch.sigmoid(x @ W[p + "g"].T)[..., None]).flatten(2) @ W[p + "o"].T
        x = x + _layer_norm(y, W[f"l{i}.norm1"], eps)
        p, f = f"l{i}.mlp.", L["mlp"]
        c, s = _shares(torch.sigmoid(x @ W[p + "router"].T), f["router"], 2)
        y = _experts(x, c, s * f["router"]["scale"], lambda e, h: torch.relu(h @ W[f"{p}e{e}.up"].T) ** 2 @ W[f"{p}e{e}.down"].T)
        x = x + _layer_norm(y, W[f"l{i}.norm2"], eps)
    return _layer_norm(x[:, -1], W["final.norm"], eps) @ W["head"].T


def _kolodra(cfg, W, ids):
    eps, (B, n) = cfg["norm"]["eps"], ids.shape
    x = W["embed"][ids]
    for i, L in enumerate(cfg["layers"]):
        h = _rms(x, eps) * (1.0 + W[f"l{i}.norm1"])
        a, r, p = L["mixer"]["left"], L["mixer"]["right"], f"l{i}.mix.left."
        v = (h @ W[p + "k"].T).view(B, n, a["kv_heads"], -1)
        q = (_rms(h @ W[p + "q"].T, eps) * W[p + "q.norm"]).view(B, n, a["heads"], -1)
        k = (_rms(v.flatten(2), eps) * W[p + "k.norm"]).view(v.shape)
        o = _attend(_rope(q, a["rot"]["base"], a["rot"]["dims"]), _rope(k, a["rot"]["base"], a["rot"]["dims"]), v, a["scale"])
        y = (o * torch.sigmoid(h @ W[p + "g"].T)[..., None]).flatten(2) @ W[p + "o"].T
        p, sh = f"l{i}.mix.right.", (B, n, r["heads"], -1)
        q, k, v = ((h @ W[p + s].T).view(sh) for s in "qkv")
        w = (torch.sigmoid((h @ W[p + "a1"].T) @ W[p + "a2"].T + W[p + "a2.b"]) ** (1.0 / r["tau"])).view(sh)
        o = _decayed(q * r["dim"] ** -0.5, k, v, lambda t: w[:, t])
        y = y + ((_rms(o, eps) * W[p + "norm"]).flatten(2) * _silu(h @ W[p + "g"].T)) @ W[p + "o"].T
        p = f"l{i}.mlp."
        g = h @ W[p + "gate"].T
        g = 0.5 * g * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (g + 0.044715 * g ** 3)))
        x = x + y + (g * (h @ W[p + "up"].T)) @ W[p + "down"].T
    cap = cfg["logit_softcap"]
    return cap * torch.tanh((_rms(x[:, -1], eps) * (1.0 + W["final.norm"])) @ W["head"].T / cap)


def _order(cfg):
    """[(layer, pass that starts with it or None)]"""
    a, z, times = (cfg["loop"][k] for k in ("start", "stop", "times"))
    body = [(i, t if i == a else None) for t in range(times) for i in range(a, z)]
    return [(i, None) for i in range(a)] + body + [(i, None) for i in range(z, len(cfg["layers"]))]


def _conv(x, w):
    taps = w.shape[1]
    full = torch.cat([x.new_zeros(x.shape[0], taps - 1, x.shape[2]), x], 1)
    return sum(full[:, j:j + x.shape[1]] * w[:, j] for j in range(taps))


def _unit(x):
    return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)


def _bibapel(cfg, W, ids):
    eps, (B, n) = cfg["norm"]["eps"], ids.shape
    g = cfg["embedding"]["bigram"]
    pair = torch.cat([torch.full_like(ids[:, :1], g["buckets"]), (ids[:, :-1] * g["mul_prev"] + ids[:, 1:] * g["mul_cur"]) % g["buckets"]], 1)
    x = x0 = W["embed"][ids] * cfg["embedding"]["scale"] + W["bigram"][pair] + W["pos"][:n]
    for i, t in _order(cfg):
        if t is not None:
            x = torch.cat([x, x0], -1) @ W["loop.in"].T + W["loop.step"][t]
        L, p = cfg["layers"][i], f"l{i}.mix."
        m, h = L["mixer"], _rms(x, eps) * W[f"l{i}.norm1"]
        if L["type"] == "attention":
            q, k, v = ((h @ W[p + s].T).view(B, n, m["heads" if s == "q" else "kv_heads"], -1) for s in "qkv")
            o = _attend(q, k, v, m["scale"], m["mask"]["size"], m["mask"]["keep_first"], sink=True).flatten(2)
        elif L["type"] == "lightning":
            q, k, v = (_silu(h @ W[p + s].T).view(B, n, m["heads"], -1) for s in "qkv")
            a = torch.tensor(m["decay"], dtype=x.dtype, device=x.device)[None, :, None]
            o = _rms(_decayed(q, k, v, lambda t: a).flatten(2), eps) * W[p + "norm"] * torch.sigmoid(h @ W[p + "g"].T)
        else:
            H, G = m["heads"], m["kv_heads"]
            q, k, v = (_silu(_conv(h @ W[p + s].T, W[p + s + ".conv"])) for s in "qkv")
            q = (_unit(q.view(B, n, G, -1)) * m["dim"] ** -0.5).repeat_interleave(H // G, 2)
            k, v = _unit(k.view(B, n, G, -1)).repeat_interleave(H // G, 2), v.view(B, n, H, -1)
            beta = torch.sigmoid(h @ W[p + "b"].T)
            w = torch.nn.functional.softplus((h @ W[p + "a1"].T) @ W[p + "a2"].T + W[p + "dt_bias"]).view(B, n, H, -1)
            w = torch.exp(-torch.exp(W[p + "A_log"])[:, None] * w)

            def step(t, S):
                S = w[:, t, :, :, None] * S
                u = beta[:, t, :, None] * (v[:, t] - (k[:, t, :, None, :] @ S)[..., 0, :])
                S = S + k[:, t, :, :, None] * u[:, :, None, :]
                return (q[:, t, :, None, :] @ S)[..., 0, :], S
            o = _scan(n, torch.zeros(B, H, q.shape[-1], v.shape[-1], dtype=x.dtype, device=x.device), step)
            o = (_rms(o, eps) * W[p + "norm"]).flatten(2) * torch.sigmoid((h @ W[p + "g1"].T) @ W[p + "g2"].T)
        y = o @ W[p + "o"].T
        p, h, lim = f"l{i}.mlp.", _rms(x, eps) * W[f"l{i}.norm2"], L["mlp"]["limit"]
        ga, u = (h @ W[p + "gate"].T).clamp(max=lim), (h @ W[p + "up"].T).clamp(-lim, lim)
        x = x + y + (ga * torch.sigmoid(1.702 * ga) * (u + 1.0)) @ W[p + "down"].T
    return (_rms(x[:, -1], eps) * W["final.norm"]) @ W["embed"].T


def _yarn(rot):
    dims, base, s = rot["dims"], rot["base"], rot["scaling"]

    def turns(t):
        return dims * math.log(s["original"] / (2.0 * math.pi * t)) / (2.0 * math.log(base))
    lo, hi = max(math.floor(turns(s["fast"])), 0), min(math.ceil(turns(s["slow"])), dims - 1)
    ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(dims // 2)]
    f = [base ** (-2.0 * i / dims) * (r / s["factor"] + 1.0 - r) for i, r in enumerate(ramp)]
    return f, 0.1 * math.log(s["factor"]) + 1.0


def _pimodra(cfg, W, ids):
    eps, parts, (B, n) = cfg["norm"]["eps"], cfg["norm"]["groups"], ids.shape

    def norm(x, w):
        return _rms(x.view(*x.shape[:-1], parts, -1), eps).view(x.shape) * w
    x = W["embed"][ids]
    for i, t in _order(cfg):
        if t is not None:
            x = x + W["loop.step"][t]
        L, p = cfg["layers"][i], f"l{i}.mix."
        m, h = L["mixer"], norm(x, W[f"l{i}.norm1"])
        q, k, v = ((h @ W[p + s].T).view(B, n, m["heads" if s == "q" else "kv_heads"], -1) for s in "qkv")
        f, gain = _yarn(m["rot"])
        q, k = (_rms(_rope(u, 0, m["rot"]["dims"], gain, f, halves=True), eps) for u in (q, k))
        o = _attend(q, k, v, m["scale"], m["mask"]["size"], talk=W[p + "talk"]).flatten(2)
        y = (o * torch.sigmoid(h @ W[p + "g"].T)) @ W[p + "o"].T
        x = x + norm(y, W[f"l{i}.norm1b"])
        p, mlp, h = f"l{i}.mlp.", L["mlp"], norm(x, W[f"l{i}.norm2"])
        if mlp["kind"] == "dense":
            u, a = h @ W[p + "up"].T, W[p + "act"]
            y = (a[0] * _rms(u, eps) + a[1] * _rms(u ** 2, eps) + a[2] * _rms(u ** 3, eps) + a[3]) @ W[p + "down"].T
        else:
            c, s = _shares(torch.softmax(h @ W[p + "router"].T, -1), mlp["router"], 1)
            y = _experts(h, c, s, lambda e, r: (_silu(r @ W[f"{p}e{e}.gate"].T) * (r @ W[f"{p}e{e}.up"].T)) @ W[f"{p}e{e}.down"].T)
        x = x + norm(y, W[f"l{i}.norm2b"])
    return norm(x[:, -1], W["final.norm"]) @ W["embed"].T


@torch.no_grad()
def exact(case, seed):
    ids = _ids(case, seed).to(DEVICE)
    if case["model"] not in STACKS:
        return _llama(case, ids).cpu()
    cfg = _config(case["model"], case["size"])
    plan = _stack_plan(cfg)
    forward = {"sekolorn": _sekolorn, "kolodra": _kolodra, "bibapel": _bibapel, "pimodra": _pimodra}[case["model"]]
    return forward(cfg, _Lazy(lambda name: _stack_tensor(plan, name).double()), ids).cpu()
