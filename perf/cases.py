"""The work that users of this framework have it do, as cases that can be timed.

Each case is one block of a gpt-oss or Qwen3 engine, called as an engine calls
it: the MoE layers of one token (decode), of a few users' tokens (a small
batch) or of a prompt (prefill), the attention block of one token, and the LM
head.  Sizes are the bench configurations' and the tests', with odd token
counts and shapes among them.  Weights and inputs have the distributions of
cpubrrr_amd.synth (k-quant scales small enough for weights of ~0.02), drawn on
the GPU from the seed alone.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from cpubrrr_amd import _lib as L
from cpubrrr_amd.attn import Attention
from cpubrrr_amd.head import LmHead
from cpubrrr_amd.moe import MoeBlock, MoeConfig

HD = 64                 # head size of the attention block
EPS = 1e-5              # rms_eps of gpt-oss; Qwen3's is 1e-6
SETS = 2                # distinct sets of expert tensors in a stack (see expert_tensors)


# ---------------------------------------------------------------- the cases
def gptoss(name, **kw):
    """gpt-oss-20b's MoE layer unless said otherwise.  chain: the layers follow each other in one
    call, on one x; otherwise each is a call of its own on an x of its own, as between an engine's
    attention blocks (and a change of rounding in one layer stays there)."""
    c = {"name": name, "kind": "gptoss", "d": 2880, "dff": 2880, "experts": 32, "top_k": 4, "layers": 1,
         "tokens": 1, "chain": False, "host": False}
    c.update(kw)
    return c


def qwen(name, **kw):
    """Qwen3-30B-A3B's MoE layer unless said otherwise (down_type 14: Q6_K, 12: Q4_K)."""
    c = {"name": name, "kind": "qwen", "d": 2048, "dff": 768, "experts": 128, "top_k": 8, "layers": 1,
         "tokens": 1, "down_type": 14, "chain": False, "host": False}
    c.update(kw)
    return c


def attn(name, **kw):
    """gpt-oss-20b's attention block, one token at position `pos`, each layer on an x of its own."""
    c = {"name": name, "kind": "attn", "d": 2880, "heads": 64, "kv_heads": 8, "window": 128, "layers": 2, "pos": 1023}
    c.update(kw)
    return c


def head(name, **kw):
    """gpt-oss-20b's LM head: `tokens` greedy tokens, and one token with its candidates' logits."""
    c = {"name": name, "kind": "head", "d": 2880, "vocab": 201088, "bits": 4, "tokens": 4}
    c.update(kw)
    return c


def listed():
    return [
        # the smallest call: one token through one small layer, from and to host memory, as the
        # engines' worker loop calls it without a device pipeline of its own
        qwen("qwen small host token", d=512, dff=512, experts=16, down_type=12, host=True),
        # decode, one user: one token through the stack, asynchronous on the engine's stream
        gptoss("gpt-oss decode", layers=6, chain=True),
        qwen("qwen decode", layers=12),
        # a few users' next tokens, or one user's drafted ones, in one batch
        gptoss("gpt-oss batch 3", layers=4, tokens=3),
        gptoss("gpt-oss batch 24", layers=2, tokens=24),
        qwen("qwen batch 11", layers=4, tokens=11, down_type=12),
        # a prompt: the bench's batch, and longer odd ones (gpt-oss-120b's 128 experts)
        gptoss("gpt-oss prefill 512", tokens=512),
        gptoss("gpt-oss-120b prefill 2049", experts=128, tokens=2049),
        qwen("qwen prefill 777", layers=2, tokens=777),
        # the attention block of one token in a short and in a long conversation
        attn("attention at 1023", layers=8, pos=1023),
        attn("attention at 7999", layers=2, pos=7999),
        # greedy tokens of four hidden states, then one for a sampler that needs the logits
        head("lm head"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gptoss"] * 5 + ["qwen"] * 4 + ["attn"] * 2 + ["head"])
    if kind == "attn":
        pos = _log_int(rng, 4, 8000)
        c = attn("", layers=rng.randint(2, 8 if pos < 2000 else 2), pos=pos)
        if rng.random() < 0.2:
            c.update(d=32 * rng.randint(16, 64), heads=16, kv_heads=4)
    elif kind == "head":
        c = head("", vocab=4 * rng.randint(8000, 50272), bits=rng.choice([4, 2]), tokens=rng.randint(1, 4))
    else:
        tokens = 1 if rng.random() < 0.25 else _log_int(rng, 2, 1500)
        layers = rng.randint(2, 6) if tokens == 1 else rng.randint(1, 3) if tokens < 48 else 1
        host = rng.random() < 0.15
        if kind == "gptoss":
            c = gptoss("", tokens=tokens, experts=rng.choice([32, 32, 128]))
            if rng.random() < 0.3:
                c.update(d=32 * rng.randint(15, 90), dff=32 * rng.randint(15, 90), experts=rng.choice([16, 32]))
            if c["experts"] == 128:
                layers = min(layers, 2)
        else:
            c = qwen("", tokens=tokens, down_type=rng.choice([14, 14, 12]))
            if rng.random() < 0.3:
                c.update(d=rng.choice([512, 1024, 4096]), dff=rng.choice([512, 768, 1536]), experts=rng.choice([32, 64]))
        c.update(layers=1 if host else layers, chain=not host and tokens == 1 and rng.random() < 0.5, host=host)
    del c["name"]
    return c


# ---------------------------------------------------------------- inputs
def _gen(seed, *what):
    """A generator on the GPU for one tensor of one case."""
    s = int(seed) & 0x7FFFFFFF
    for w in what:
        s = (s * 1000003 + w + 1) % (1 << 61)
    return torch.Generator(device="cuda").manual_seed(s)


def _normal(shape, sigma, seed, *what):
    return torch.randn(shape, generator=_gen(seed, *what), device="cuda") * sigma


def _bytes(shape, seed, *what):
    return torch.randint(0, 256, shape, generator=_gen(seed, *what), device="cuda", dtype=torch.uint8)


def _mxfp4(rows, cols, seed, *what):
    """[rows][cols / 32][17]: codes uniform, e8m0 = 127 + U{-6 .. -3}."""
    w = _bytes((rows, cols // 32, 17), seed, *what)
    w[..., 0] = torch.randint(121, 125, w.shape[:2], generator=_gen(seed, 77, *what), device="cuda", dtype=torch.uint8)
    return w


def _half_bytes(shape, sigma, seed, *what):
    return _normal(shape, sigma, seed, *what).abs().half().unsqueeze(-1).view(torch.uint8)


def _q4k(rows, cols, seed, *what):
    w = _bytes((rows, cols // 256, 144), seed, *what)
    w[..., 0:2] = _half_bytes(w.shape[:2], 1e-4, seed, 78, *what)      # d
    w[..., 2:4] = _half_bytes(w.shape[:2], 5e-4, seed, 79, *what)      # dmin
    return w


def _q6k(rows, cols, seed, *what):
    w = _bytes((rows, cols // 256, 210), seed, *what)
    w[..., 208:210] = _half_bytes(w.shape[:2], 2e-5, seed, 80, *what)  # d
    return w


def expert_tensors(c, seed, which):
    """Gate, up and down of every expert, native GGUF rows.  A stack's layers
    take SETS of them in turn, each layer loaded to memory of its own: the
    routers differ from layer to layer, and what a layer reads does not depend
    on another's bytes."""
    ne, d, ff = c["experts"], c["d"], c["dff"]
    if c["kind"] == "gptoss":
        return {"gate": _mxfp4(ne * ff, d, seed, which, 1), "up": _mxfp4(ne * ff, d, seed, which, 2),
                "down": _mxfp4(ne * d, ff, seed, which, 3),
                "gate_b": _normal((ne, ff), 0.01, seed, which, 4), "up_b": _normal((ne, ff), 0.01, seed, which, 5),
                "down_b": _normal((ne, d), 0.01, seed, which, 6)}
    down = _q6k if c["down_type"] == 14 else _q4k
    return {"gate": _q4k(ne * ff, d, seed, which, 1), "up": _q4k(ne * ff, d, seed, which, 2),
            "down": down(ne * d, ff, seed, which, 3)}


def router_tensors(c, seed, layer):
    ne, d = c["experts"], c["d"]
    r = {"router_w": _normal((ne, d), 0.02, seed, 100 + layer, 1), "norm_w": 1.0 + _normal((d,), 0.05, seed, 100 + layer, 2)}
    if c["kind"] == "gptoss":
        # expert load skewed as Zipf(1.1) over a random order of the experts
        rank = torch.randperm(ne, generator=_gen(seed, 100 + layer, 3), device="cuda").double() + 1
        r["router_b"] = (-1.1 * rank.log() - torch.logsumexp(-1.1 * rank.log(), 0)).float()
    return r


def moe_input(c, seed):
    return _normal((1 if c["chain"] else c["layers"], c["tokens"], c["d"]), 1.0, seed, 9)


def attn_tensors(c, seed, layer):
    d, nq, nkv = c["d"], c["heads"] * HD, c["kv_heads"] * HD
    t = {"attn_norm": 1.0 + _normal((d,), 0.05, seed, 200 + layer, 1)}
    for i, (k, shape) in enumerate((("wq", (nq, d)), ("wk", (nkv, d)), ("wv", (nkv, d)), ("wo", (d, nq)))):
        t[k] = _normal(shape, 0.02, seed, 200 + layer, 2 + i).bfloat16()
    for i, (k, n, sigma) in enumerate((("bq", nq, 0.01), ("bk", nkv, 0.01), ("bv", nkv, 0.01), ("bo", d, 0.01),
                                       ("sinks", c["heads"], 1.0))):
        t[k] = _normal((n,), sigma, seed, 200 + layer, 6 + i)
    return t


def attn_past(c, seed, layer):
    """Hidden states of the positions before the timed one."""
    return _normal((c["pos"], c["d"]), 1.0, seed, 300 + layer)


def attn_input(c, seed):
    return _normal((c["layers"], c["d"]), 1.0, seed, 9)


def head_tensors(c, seed):
    # the hidden states lean towards a few rows, as a trained model's do
    w = _normal((c["vocab"], c["d"]), 0.02, seed, 400, 1).bfloat16()
    norm = 1.0 + _normal((c["d"],), 0.05, seed, 400, 2)
    x = _normal((c["tokens"] + 1, c["d"]), 1.0, seed, 400, 3)
    at = torch.randint(0, c["vocab"], (c["tokens"] + 1,), generator=_gen(seed, 400, 4), device="cuda")
    return w, norm, x + 10.0 * w[at].float()


def _np(t):
    return (t.view(torch.int16).cpu().numpy().view(np.uint16) if t.dtype == torch.bfloat16 else t.cpu().numpy())


# ---------------------------------------------------------------- prepare and run
_STREAM = None


def _stream():
    """The one stream of the program that the handles work on."""
    global _STREAM
    if _STREAM is None:
        _STREAM = torch.cuda.Stream()
    return _STREAM


def _prepare_moe(c, seed):
    kw = dict(d=c["d"], n_expert=c["experts"], top_k=c["top_k"], d_ff=c["dff"], n_layer=c["layers"], max_tokens=c["tokens"])
    cfg = MoeConfig.gptoss(**kw) if c["kind"] == "gptoss" else MoeConfig.qwen3(down_type=c["down_type"], **kw)
    blk = MoeBlock(cfg)
    for which in range(min(SETS, c["layers"])):
        shared = {k: _np(t) for k, t in expert_tensors(c, seed, which).items()}
        for layer in range(which, c["layers"], SETS):
            blk.load_layer(layer, {**shared, **{k: _np(t) for k, t in router_tensors(c, seed, layer).items()}})
    x0 = moe_input(c, seed)
    s = {"moe": blk}
    if c["host"]:
        s["x_host"] = (x0[0] if c["tokens"] > 1 else x0[0, 0]).cpu().numpy()
    else:
        blk.set_stream(_stream().cuda_stream)
        s["x0"], s["x"] = x0, torch.empty_like(x0)
    return s


def _prepare_attn(c, seed):
    at = Attention(c["d"], c["heads"], c["kv_heads"], c["layers"], max_seq=c["pos"] + 1, sliding_window=c["window"])
    at.set_stream(_stream().cuda_stream)
    for layer in range(c["layers"]):
        at.load_layer(layer, {k: _np(t) for k, t in attn_tensors(c, seed, layer).items()})
        past = attn_past(c, seed, layer)
        torch.cuda.synchronize()
        for p in range(c["pos"]):
            at.forward_device(layer, p, past[p].data_ptr())
        at.sync()
    x0 = attn_input(c, seed)
    return {"attn": at, "x0": x0, "x": torch.empty_like(x0)}


def _prepare_head(c, seed):
    w, norm, x = head_tensors(c, seed)
    h = LmHead(c["d"], c["vocab"])
    h.load(_np(w), _np(norm))
    h.set_screen(c["bits"])
    h.set_stream(_stream().cuda_stream)
    nc = h.cfg.n_slices * h.cfg.n_cand
    s = {"head": h, "x": x[:-1].contiguous(), "tokens": torch.zeros(c["tokens"], dtype=torch.int32, device="cuda"),
         "x_host": x[-1].cpu().numpy(), "cand_ids": np.zeros(nc, np.int32), "cand_logits": np.zeros(nc, np.float32)}
    s["trace"] = L.HeadTrace(cand_ids=s["cand_ids"].ctypes.data_as(L.i32p), cand_logits=s["cand_logits"].ctypes.data_as(L.f32p))
    return s


def prepare(case, seed):
    c = case
    make = {"gptoss": _prepare_moe, "qwen": _prepare_moe, "attn": _prepare_attn, "head": _prepare_head}[c["kind"]]
    s = make(c, seed)
    s["case"] = c
    torch.cuda.synchronize()
    return s


def run(state):
    c = state["case"]
    if c["kind"] in ("gptoss", "qwen"):
        if c["host"]:
            return state["moe"].forward(0, state["x_host"])[0]
        with torch.cuda.stream(_stream()):
            state["x"].copy_(state["x0"])            # the embedding, or the block before, writes x
        if c["chain"]:
            state["moe"].forward_device(0, c["layers"], state["x"].data_ptr(), c["tokens"])
        else:
            for layer in range(c["layers"]):
                state["moe"].forward_device(layer, 1, state["x"][layer].data_ptr(), c["tokens"])
        return state["x"]
    if c["kind"] == "attn":
        with torch.cuda.stream(_stream()):
            state["x"].copy_(state["x0"])
        for layer in range(c["layers"]):
            state["attn"].forward_device(layer, c["pos"], state["x"][layer].data_ptr())
        return state["x"]
    h = state["head"]
    for i in range(c["tokens"]):
        h.forward_device(state["x"][i].data_ptr(), state["tokens"][i:].data_ptr())
    chosen = C.c_int32()
    L.check(L.lib().cpb_head_forward(h._h, state["x_host"].ctypes.data_as(L.f32p), C.byref(chosen),
                                     C.byref(state["trace"])), "cpb_head_forward")
    return {"tokens": state["tokens"], "chosen": int(chosen.value), "cand_ids": state["cand_ids"],
            "cand_logits": state["cand_logits"]}


# ---------------------------------------------------------------- work and tolerance
def work(case):
    c = case
    if c["kind"] in ("gptoss", "qwen"):
        n, d, ff, ne, k = c["tokens"], c["d"], c["dff"], c["experts"], c["top_k"]
        used = ne * (1.0 - (1.0 - k / ne) ** n)      # experts that some token takes, were all as likely
        if c["kind"] == "gptoss":
            expert = (2 * ff * d + d * ff) * 17 / 32 + 4 * (2 * ff + d)
        else:
            expert = 2 * ff * d * 144 / 256 + d * ff * (210 if c["down_type"] == 14 else 144) / 256
        return {"bytes": c["layers"] * (used * expert + 4 * ne * d + 8 * n * d),
                "flops": c["layers"] * 2.0 * n * (3 * k * d * ff + ne * d)}
    if c["kind"] == "attn":
        d, nq, nkv = c["d"], c["heads"] * HD, c["kv_heads"] * HD
        rows = (nq + 2 * nkv) * d + d * nq
        seen = [min(c["pos"] + 1, c["window"]) if layer % 2 == 0 else c["pos"] + 1 for layer in range(c["layers"])]
        return {"bytes": c["layers"] * (rows * 36 / 32 + 8 * d) + sum(seen) * nkv * 8.0,
                "flops": c["layers"] * 2.0 * rows + sum(seen) * 4.0 * nq}
    b = 18 if c["bits"] == 4 else 10
    calls = c["tokens"] + 1
    return {"bytes": calls * (c["vocab"] * c["d"] * b / 32.0 + 4 * c["d"]), "flops": calls * 2.0 * c["vocab"] * c["d"]}


def tolerance(case):
    # Sums in another order move the activations by ~1e-7, which now and then moves one 8-bit
    # activation by a quantum (1/127 of its block's largest).  Measured against exact(): up to
    # 2e-4 of the result in one MoE layer and one attention block; 1e-2 after some layers of a
    # chain, each of which quantises what the last one changed; in the head up to 6e-3, where two
    # candidates change places.
    if case["kind"] == "head":
        return {"rel": 2e-2, "max": 0.5, "differ": 0.01}
    if case["kind"] != "attn" and case["chain"]:
        return {"rel": 3e-2, "max": 0.5}
    return {"rel": 1e-3, "max": 2e-2}


# ---------------------------------------------------------------- the same in 64 bits
E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _deq_mxfp4(w):
    v = torch.tensor(E2M1 + [-e for e in E2M1], dtype=torch.float64, device=w.device)
    q = torch.cat([w[..., 1:] & 15, w[..., 1:] >> 4], -1).long()
    return (v[q] * torch.exp2(w[..., :1].double() - 127)).flatten(-2)


def _half(b):
    return b.contiguous().view(torch.float16).double()


def _deq_q4k(w):
    d, dmin, s = _half(w[..., 0:2]), _half(w[..., 2:4]), w[..., 4:16].long()
    sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | (s[..., 0:4] >> 6 << 4)], -1)
    mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | (s[..., 4:8] >> 6 << 4)], -1)
    q = w[..., 16:].unflatten(-1, (4, 1, 32))
    q = torch.cat([q & 15, q >> 4], -2).flatten(-3, -2).double()        # [..., 8, 32]
    return ((d * sc).unsqueeze(-1) * q - (dmin * mn).unsqueeze(-1)).flatten(-3)


def _deq_q6k(w):
    ql, qh = w[..., :128].unflatten(-1, (2, 2, 32)), w[..., 128:192].unflatten(-1, (2, 1, 32))
    low = torch.stack([ql[..., 0, :] & 15, ql[..., 1, :] & 15, ql[..., 0, :] >> 4, ql[..., 1, :] >> 4], -2)
    high = torch.cat([qh & 3, qh >> 2 & 3, qh >> 4 & 3, qh >> 6], -2)
    q = (low | high << 4).double() - 32                                   # [..., 2, 4, 32]
    sc = w[..., 192:208].contiguous().view(torch.int8).double().unflatten(-1, (2, 4, 2, 1))
    d = _half(w[..., 208:210]).unsqueeze(-1).unsqueeze(-1).unsqueeze(-1)
    return (d * sc * q.unflatten(-1, (2, 16))).flatten(-5)


def _q8(x, block):
    """Symmetric 8-bit blocks with a real scale, ties away from zero: MXFP4's and Q8_0's activations."""
    b = x.unflatten(-1, (-1, block))
    sc = b.abs().amax(-1, keepdim=True).clamp_min(1e-12) / 127
    r = b / sc
    return ((r.sign() * (r.abs() + 0.5).floor()).clamp(-127, 127) * sc).flatten(-2)


def _q8_rows(w):
    """8-bit weight rows of bf16 ones.  The codes and the 32-bit scales are what the layer stores,
    and a bf16 weight is often halfway between two codes, so these are formed in 32 bits as there."""
    b = w.float().unflatten(-1, (-1, 32))
    sc = b.abs().amax(-1, keepdim=True).clamp_min(1e-12)
    sc = sc / torch.full_like(sc, 127.0)            # a true division: by a constant it would be a product
    r = b / sc
    return ((r.sign() * (r.abs() + 0.5).floor()).clamp(-127, 127).double() * sc.double()).flatten(-2)


def _rmsnorm(x, w, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w.double()


def _exact_moe(c, seed):
    gpt = c["kind"] == "gptoss"
    ne, k, d, ff = c["experts"], c["top_k"], c["d"], c["dff"]
    block = 32 if gpt else 256
    deq = _deq_mxfp4 if gpt else _deq_q4k
    deq_down = _deq_mxfp4 if gpt else _deq_q6k if c["down_type"] == 14 else _deq_q4k
    start = moe_input(c, seed).double()
    sets = [expert_tensors(c, seed, which) for which in range(min(SETS, c["layers"]))]
    done = []
    for layer in range(c["layers"]):
        t, r = sets[layer % SETS], router_tensors(c, seed, layer)
        x = done[-1] if c["chain"] and done else start[layer]
        xn = _rmsnorm(x, r["norm_w"], EPS if gpt else 1e-6)
        logits = xn @ r["router_w"].double().T + (r["router_b"].double() if gpt else 0.0)
        top, ids = logits.topk(k, -1)
        wts = torch.softmax(top, -1)
        xq = _q8(xn, block)
        for e in ids.unique().tolist():
            tok, slot = (ids == e).nonzero(as_tuple=True)
            part = {n: t[n].unflatten(0, (ne, -1))[e] for n in ("gate", "up", "down")}
            g, u = xq[tok] @ deq(part["gate"]).T, xq[tok] @ deq(part["up"]).T
            if gpt:
                g, u = (g + t["gate_b"][e]).clamp(max=7.0), (u + t["up_b"][e]).clamp(-7.0, 7.0)
                h = g * torch.sigmoid(1.702 * g) * (u + 1)
            else:
                h = g * torch.sigmoid(g) * u
            y = _q8(h, block) @ deq_down(part["down"]).T
            if gpt:
                y = y + t["down_b"][e]
            x = x.index_add(0, tok, wts[tok, slot].unsqueeze(-1) * y)
        done.append(x)
    if c["host"]:
        return x if c["tokens"] > 1 else x[0]
    return x[None] if c["chain"] else torch.stack(done)


def _rope(v, pos):
    """YaRN as gpt-oss sets it (factor 32 from 4096 positions); the angles are the path's own
    32-bit ones, which are part of its definition, their sine and cosine exact."""
    i = torch.arange(HD // 2, device=v.device, dtype=torch.float32)
    base = 150000.0
    low = max(math.floor(HD * math.log(4096 / (32 * 2 * math.pi)) / (2 * math.log(base))), 0)
    high = min(math.ceil(HD * math.log(4096 / (2 * math.pi)) / (2 * math.log(base))), HD - 1)
    ex = pos.float()[:, None] * torch.pow(torch.tensor(base, device=v.device), -(2 * i) / HD)
    mix = 1 - ((i - low) / max(high - low, 0.001)).clamp(0, 1)
    theta = (ex / 32 * (1 - mix) + ex * mix).double()[:, None]
    m = 1.0 + 0.1 * math.log(32.0)
    cos, sin = theta.cos() * m, theta.sin() * m
    a, b = v[..., :HD // 2], v[..., HD // 2:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _exact_attn(c, seed):
    nh, nkv, pos = c["heads"], c["kv_heads"], c["pos"]
    start_x, done = attn_input(c, seed).double(), []
    at = torch.arange(pos + 1, device="cuda")
    for layer in range(c["layers"]):
        x, t = start_x[layer], attn_tensors(c, seed, layer)
        w = {k: _q8_rows(t[k]) for k in ("wq", "wk", "wv", "wo")}
        start = max(0, pos - c["window"] + 1) if layer % 2 == 0 else 0
        xs = torch.cat([attn_past(c, seed, layer)[start:].double(), x[None]])
        xq = _q8(_rmsnorm(xs, t["attn_norm"], EPS), 32)
        q = _rope((xq[-1:] @ w["wq"].T + t["bq"]).unflatten(-1, (nh, HD)), at[-1:])[0]
        k = _rope((xq @ w["wk"].T + t["bk"]).unflatten(-1, (nkv, HD)), at[start:])
        v = (xq @ w["wv"].T + t["bv"]).unflatten(-1, (nkv, HD))
        out = []
        for h in range(nh):
            g = h // (nh // nkv)
            s = torch.cat([k[:, g] @ q[h] / math.sqrt(HD), t["sinks"][h:h + 1].double()])
            out.append(torch.softmax(s, 0)[:-1] @ v[:, g])
        done.append(x + _q8(torch.cat(out), 32) @ w["wo"].T + t["bo"])
    return torch.stack(done)


def _q4_screen_rows(w):
    """The 4-bit rows of the screen: per 32 values the bf16 scale of 17 (largest value / -(7 .. 8))
    with the least squared error."""
    v = w.float().unflatten(-1, (-1, 32))
    vmax = v.gather(-1, v.abs().argmax(-1, keepdim=True))
    best, err = torch.zeros_like(v), torch.full_like(vmax, float("inf"))
    for t in range(17):
        d = (vmax / -(7.0 + t / 16)).bfloat16().float()
        y = ((v / d + 8.5).floor().clamp(0, 15) - 8) * d
        e = (v - y).square().sum(-1, keepdim=True)
        best, err = torch.where(e < err, y, best), torch.minimum(e, err)
    return best.flatten(-2).double()


def _q2_screen_rows(w):
    v = w.float().unflatten(-1, (-1, 32))
    d = (v.gather(-1, v.abs().argmax(-1, keepdim=True)) / -2.0).bfloat16().float()
    return (((v / d + 2.5).floor().clamp(0, 3) - 2) * d).flatten(-2).double()


def _exact_head(c, seed):
    """The candidates' logits: of each of twelve slices of the vocabulary (as even as quads of rows
    allow) the eight rows that the screen ranks first.  Where a rank is decided in the last bits
    the two lists may differ in a place."""
    w, norm, x = head_tensors(c, seed)
    xq = _q8(_rmsnorm(x[-1].double(), norm, EPS), 32)
    rows = _q4_screen_rows if c["bits"] == 4 else _q2_screen_rows
    screen = torch.cat([rows(p) @ xq for p in w.split(8192)])
    quads, logits = c["vocab"] // 4, []
    for s in range(12):
        a, b = 4 * (quads * s // 12), 4 * (quads * (s + 1) // 12)
        ids = a + screen[a:b].topk(8).indices
        logits.append(_q8_rows(w[ids]) @ xq)
    return {"tokens": None, "chosen": None, "cand_ids": None, "cand_logits": torch.cat(logits)}


def exact(case, seed):
    c = case
    if c["kind"] == "attn":
        return _exact_attn(c, seed)
    return _exact_head(c, seed) if c["kind"] == "head" else _exact_moe(c, seed)
