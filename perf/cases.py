"""The work that a user of this framework has it do, as cases that can be timed and checked.

Two levels, as in include/mllm.h: the operators on device pointers (an MLP
block put together from them, the lm_head with its argmax, the GEMVs of each
storage, a layer stack in one launch, the dequantiser) and the engine (prompts,
chained and stepwise decode, the rows of a speculation pass) on models of the
repository's own configurations, with the weights drawn on the GPU.

    listed()           the named cases
    draw(rng)          another case of the same ranges
    prepare(case, s)   weights, inputs and handles from the seed s
    run(state)         one pass through the public entry points
    work(case)         the bytes and operations a pass cannot do without
    tolerance(case)    how far another correct implementation may be off
    exact(case, s)     what run() returns, in 64 bits, by plain torch
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "microllm-lab_amd"))

import mllm  # noqa: E402
from mllm import abi, pgw  # noqa: E402

DEV = "cuda"
GROUP = 32
EPS = 1e-6  # infer.js:8


# ---------------------------------------------------------------- the cases
def _model(op, base, kind="q4", **kw):
    c = pgw.CONFIGS[base]
    m = {"op": op, "arch": c.arch, "kind": kind, "group": GROUP, "vocab": c.vocab_size, "layers": c.n_layers,
         "d_model": c.d_model, "heads": c.n_heads, "kv_heads": c.n_kv_heads, "d_ff": c.d_ff,
         "max_seq": c.max_seq_len, "kv_fp16": False}
    m.update(kw)
    return m


def listed():
    return [
        # the operators as a host drives them at decode: one token's MLP block
        # of the 135M shape (five small launches)
        dict(name="mlp_ops_1x576", op="mlp_ops", tokens=1, d_model=576, d_ff=1536),
        # the same operators over a prompt (gemmGeneric), 360M shape, odd length
        dict(name="mlp_ops_301x960", op="mlp_ops", tokens=301, d_model=960, d_ff=2560),
        # the last GEMV of every greedy token: 360M lm_head and its argmax
        dict(name="head_argmax_q4", op="argmax", rows=49152, cols=960),
        # an unquantised lm_head (135M shape) through the f32 operator
        dict(name="gemv_f32_head", op="gemv", fmt="f32", rows=49152, cols=576),
        # the gate rows of a 32-layer stack in one launch, Q8 group-32
        dict(name="stack_q8g32", op="stack", fmt="q8g32", count=32, rows=2560, cols=960),
        # the embedding table de-quantised for a consumer of plain floats
        dict(name="dequant_q4_head", op="dequant", rows=49152, cols=576),
        # chat decode: chained greedy tokens after a short prompt, then logits
        dict(_model("chain", "smollm2-135m", ctx=32, steps=16), name="chain_q4_135m"),
        # a long prompt with the f16 cache (360M, 1536 tokens)
        dict(_model("prompt", "smollm2-360m", kv_fp16=True, tokens=1536), name="prompt_q4_360m_1536"),
        # a short prompt, odd length: time to first token (GPT-2)
        dict(_model("prompt", "gpt2-124m", tokens=33), name="prompt_q4_gpt2_33"),
        # prompt-lookup speculation: a token and four drafts at context 512
        dict(_model("verify", "smollm2-135m", ctx=512, steps=5), name="verify_q4_135m_5"),
        # stepwise decode (logits to the host each token) of a per-row Q8 model
        dict(_model("step", "smollm2-135m", kind="q8", ctx=700, steps=4), name="step_q8_135m"),
        # a prompt of an f16 model
        dict(_model("prompt", "smollm2-135m", kind="f16", tokens=200), name="prompt_f16_135m_200"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["mlp_ops", "argmax", "gemv", "stack", "dequant", "chain", "prompt", "prompt", "verify", "step"])
    cols = 32 * _log(rng, 4, 96)
    if op == "mlp_ops":
        return dict(op=op, tokens=_log(rng, 1, 400), d_model=64 * rng.randint(2, 16), d_ff=32 * rng.randint(8, 80))
    if op == "argmax":
        return dict(op=op, rows=_log(rng, 1000, 51000), cols=min(cols, 1024))
    if op == "gemv":
        fmt = rng.choice(["q4", "q8", "q8g32", "f32"])
        rows = _log(rng, 200, 50000)
        cols = min(cols, max(128, 32 * int(900000 / rows)))
        return dict(op=op, fmt=fmt, rows=rows, cols=cols - (rng.randint(0, 3) if fmt == "f32" else 0))
    if op == "stack":
        return dict(op=op, fmt=rng.choice(["q4", "q8g32"]), count=rng.randint(2, 32), rows=_log(rng, 64, 2560),
                    cols=min(cols, 2560))
    if op == "dequant":
        return dict(op=op, rows=_log(rng, 100, 50000), cols=min(cols, 1024))
    # engine: shapes between the tests' small ones and the configurations
    arch = rng.choice(["llama", "llama", "gpt2"])
    kv = rng.choice([1, 2, 3, 5])
    rep = 1 if arch == "gpt2" else rng.choice([1, 2, 3, 4])
    while kv * rep * 64 > 960:
        kv -= 1
    heads = rng.randint(1, 12) if arch == "gpt2" else kv * rep
    kind, group = rng.choice([("q4", 32), ("q4", 32), ("q4", 64), ("q8", 32), ("q8g32", 32), ("f16", 32),
                              ("bf16", 32), ("f32", 32)])
    c = dict(op=op, arch=arch, kind=kind, group=group, vocab=_log(rng, 500, 50000), layers=rng.randint(2, 12),
             d_model=64 * heads, heads=heads, kv_heads=heads if arch == "gpt2" else kv, d_ff=64 * rng.randint(4, 40),
             max_seq=1024, kv_fp16=rng.random() < 0.5)
    if arch == "gpt2" and op in ("chain", "verify"):
        c["op"] = op = "step"  # the chain's penalised argmax and speculation are not GPT-2's
    if op == "prompt":
        c["tokens"] = _log(rng, 2, 900 if (kind, group) == ("q4", 32) else 200)
    else:
        c["ctx"] = _log(rng, 8, 900)
        c["steps"] = rng.randint(2, 9) if op == "verify" else rng.randint(2, 24) if op == "chain" else rng.randint(1, 6)
    return c


# ---------------------------------------------------------------- weights
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * std


def _spans(w, group, top):
    """Groups of a matrix and their scales max|x| / top (1 for a zero group)."""
    ch = w.reshape(w.shape[0], -1, group)
    amax = ch.abs().amax(-1).double()
    sc = torch.where(amax > 0, amax / top, torch.ones_like(amax)).float()
    return ch, sc


def _store(w, kind, group=GROUP):
    """(data, scales) of a matrix in its storage, as the converters quantise."""
    r, c = w.shape
    if kind == "q4":
        ch, sc = _spans(w, group, 8.0)
        q = (torch.round(ch / sc[..., None]) + 8).clamp(0, 15).to(torch.uint8)
        return (q[..., 0::2] | (q[..., 1::2] << 4)).reshape(r, c // 2).contiguous(), sc
    if kind in ("q8", "q8g32"):
        ch, sc = _spans(w, c if kind == "q8" else 32, 127.0)
        q = torch.round(ch / sc[..., None]).clamp(-127, 127).to(torch.int8)
        return q.reshape(r, c).contiguous(), sc
    if kind == "f16":
        return w.to(torch.float16), None
    if kind == "bf16":
        return w.to(torch.bfloat16), None
    return w.contiguous(), None


def _plain(data, sc, kind, group=GROUP):
    """A stored matrix in 64 bits."""
    if kind == "q4":
        q = torch.stack([data & 15, data >> 4], -1).reshape(data.shape[0], -1).double() - 8.0
        return (q.reshape(q.shape[0], -1, group) * sc.double()[..., None]).reshape(q.shape)
    if kind in ("q8", "q8g32"):
        q = data.double()
        return (q.reshape(q.shape[0], sc.shape[1], -1) * sc.double()[..., None]).reshape(q.shape)
    return data.double()


def _tensors(c, seed):
    """The model's tensors in the converters' order: (name, data, scales, storage)."""
    g = _gen(seed)
    D, FF, kvd = c["d_model"], c["d_ff"], 64 * c["kv_heads"]

    def mat(name, rows, cols, std=0.02):
        data, sc = _store(_normal(g, (rows, cols), std), c["kind"], c["group"])
        return name, data, sc, c["kind"]

    def vec(name, *parts):
        return name, torch.cat(parts) if len(parts) > 1 else parts[0], None, "f32"

    def gain():
        return 1.0 + _normal(g, (D,), 0.1)

    if c["arch"] == "gpt2":
        sf = torch.exp(_normal(g, (D,), 0.1))
        yield vec("scale_factors", sf)
        yield mat("lm_head", c["vocab"], D)
        yield "wpe", _normal(g, (c["max_seq"], D), 0.02), None, "f32"
        yield vec("ln_f", gain(), _normal(g, (D,), 0.02))
        for i in range(c["layers"]):
            b = "blocks.%d." % i
            yield vec(b + "ln1", gain(), _normal(g, (D,), 0.02))
            yield mat(b + "attn.qkv", 3 * D, D)
            yield vec(b + "attn.qkv_bias", _normal(g, (3 * D,), 0.02))
            yield mat(b + "attn.proj", D, D)
            yield vec(b + "attn.proj_bias", _normal(g, (D,), 0.02))
            yield vec(b + "ln2", gain(), _normal(g, (D,), 0.02))
            yield mat(b + "mlp.fc", FF, D)
            yield vec(b + "mlp.fc_bias", _normal(g, (FF,), 0.02))
            yield mat(b + "mlp.proj", D, FF)
            yield vec(b + "mlp.proj_bias", _normal(g, (D,), 0.02))
        return
    yield mat("lm_head", c["vocab"], D)
    for i in range(c["layers"]):
        b = "blocks.%d." % i
        yield vec(b + "norm1", gain())
        yield mat(b + "attn.qkv", D + 2 * kvd, D)
        yield mat(b + "attn.proj", D, D)
        yield vec(b + "norm2", gain())
        yield mat(b + "mlp.w1", FF, D)
        yield mat(b + "mlp.w3", FF, D)
        yield mat(b + "mlp.w2", D, FF)
    yield vec("norm_f", gain())


def _bundle(c, seed):
    """The model as parse_pgw gives it: one host buffer, every blob on a
    16-byte boundary."""
    table, blobs, at = {}, [], 0

    def put(t):
        nonlocal at
        b = t.contiguous().reshape(-1).view(torch.uint8)
        off, at = at, at + b.numel() + (-b.numel() % 16)
        blobs.append(b)
        if at - off > b.numel():
            blobs.append(torch.zeros(at - off - b.numel(), dtype=torch.uint8, device=DEV))
        return off, b.numel()

    for name, data, sc, storage in _tensors(c, seed):
        shape = list(data.shape)
        if storage == "q4":
            shape[1] *= 2
        e = {"name": name, "shape": shape, "kind": c["kind"], "storage": storage, "group": c["group"]}
        if sc is not None:
            e["scaleOffset"], e["scaleNbytes"] = put(sc)
        e["offset"], e["nbytes"] = put(data)
        table[name] = e
    cfg = pgw.Config(c["arch"], c["vocab"], c["layers"], c["d_model"], c["heads"], c["kv_heads"], c["d_ff"],
                     c["max_seq"], GROUP, 100000.0 if c["arch"] == "llama" else 10000.0, 1.0)
    return pgw.Bundle(c["kind"], cfg, table, torch.cat(blobs).cpu().numpy(), 0, list(table))


def _ids(c, seed):
    """The prompt, and the tokens that follow it."""
    r = np.random.default_rng(seed)
    n = c["tokens"] if c["op"] == "prompt" else c["ctx"]
    return ([int(v) for v in r.integers(0, c["vocab"], n)], [int(v) for v in r.integers(0, c["vocab"], c.get("steps", 0))])


# ---------------------------------------------------------------- prepare and run
def _op_inputs(c, seed):
    g = _gen(seed)
    op = c["op"]
    if op == "mlp_ops":
        D, FF, T = c["d_model"], c["d_ff"], c["tokens"]
        return dict(x=_normal(g, (T, D)), gain=1.0 + _normal(g, (D,), 0.1), w1=_store(_normal(g, (FF, D), 0.02), "q4"),
                    w3=_store(_normal(g, (FF, D), 0.02), "q4"), w2=_store(_normal(g, (D, FF), 0.02), "q4"))
    if op == "stack":
        return dict(w=[_store(_normal(g, (c["rows"], c["cols"]), 0.02), c["fmt"]) for _ in range(c["count"])],
                    x=[_normal(g, (c["cols"],)) for _ in range(c["count"])])
    fmt = c.get("fmt", "q4")
    return dict(w=_store(_normal(g, (c["rows"], c["cols"]), 0.02), fmt), x=_normal(g, (c["cols"],)))


def _p(t):
    return t.data_ptr()


def prepare(case, seed):
    c = case
    if "layers" in c:
        g = mllm.PetitGPT(_bundle(c, seed), norm_eps=EPS, kv_fp16=c["kv_fp16"])
        ids, more = _ids(c, seed)
        if c["op"] != "prompt":
            g.forwardPrompt(ids)
        return dict(case=c, g=g, ids=ids, more=more)
    s = _op_inputs(c, seed)
    s["case"] = c
    f32 = dict(device=DEV, dtype=torch.float32)
    if c["op"] == "mlp_ops":
        T, D, FF = c["tokens"], c["d_model"], c["d_ff"]
        s.update(n=torch.empty(T, D, **f32), a=torch.empty(T, FF, **f32), b=torch.empty(T, FF, **f32),
                 y=torch.empty(T, D, **f32))
    elif c["op"] == "stack":
        s["y"] = [torch.empty(c["rows"], **f32) for _ in range(c["count"])]
        s["ptrs"] = [torch.tensor([_p(t) for t in v], dtype=torch.int64, device=DEV)
                     for v in ([w[0] for w in s["w"]], [w[1] for w in s["w"]], s["x"], s["y"])]
    elif c["op"] == "dequant":
        s["y"] = torch.empty(c["rows"], c["cols"], **f32)
    else:
        s["y"] = torch.empty(c["rows"], **f32)
        s["id"] = torch.zeros(1, dtype=torch.int32, device=DEV)
    return s


def run(s):
    c = s["case"]
    op = c["op"]
    if op in ("chain", "prompt", "verify", "step"):
        g = s["g"]
        if op == "prompt":
            return g.forwardPrompt(s["ids"]).copy()
        g.cacheLen = len(s["ids"])
        if op == "chain":
            out = g.decodeChain(s["more"][0], c["steps"])
            return {"ids": np.asarray(out, np.int64), "logits": g.forwardDecode(out[-1]).copy()}
        if op == "verify":
            rows, logits = g.forwardVerify(s["more"], want_logits=True)
            return {"ids": np.asarray(rows, np.int64), "logits": logits}
        return np.stack([g.forwardDecode(t).copy() for t in s["more"]])
    st = torch.cuda.current_stream().cuda_stream
    if op == "mlp_ops":
        T, D, FF = c["tokens"], c["d_model"], c["d_ff"]
        abi.call("mllm_rms_norm", D, _p(s["x"]), _p(s["gain"]), _p(s["n"]), T, EPS, st)
        for w, x, y, m, k in (("w1", "n", "a", FF, D), ("w3", "n", "b", FF, D), (None,) * 5, ("w2", "a", "y", D, FF)):
            if w is None:
                abi.call("mllm_silu_mul", T * FF, _p(s["a"]), _p(s["b"]), st)
            elif T == 1:
                abi.call("mllm_gemv_q4", m, k, _p(s[w][0]), _p(s[w][1]), GROUP, _p(s[x]), _p(s[y]), st)
            else:
                abi.call("mllm_gemm_q4", T, m, k, _p(s[w][0]), _p(s[w][1]), GROUP, _p(s[x]), _p(s[y]), st)
        return {"n": s["n"], "h": s["a"], "y": s["y"]}
    m, n = c["rows"], c["cols"]
    if op == "argmax":
        abi.call("mllm_gemv_q4_argmax", m, n, _p(s["w"][0]), _p(s["w"][1]), GROUP, _p(s["x"]), _p(s["y"]), _p(s["id"]), st)
        return {"y": s["y"], "id": s["id"]}
    if op == "dequant":
        abi.call("mllm_dequant_q4", m, n, _p(s["w"][0]), _p(s["w"][1]), GROUP, _p(s["y"]), st)
        return s["y"]
    if op == "stack":
        fn = "mllm_gemv_q4_batched" if c["fmt"] == "q4" else "mllm_gemv_q8_g32_batched"
        abi.call(fn, c["count"], m, n, *[_p(t) for t in s["ptrs"]], st)
        return s["y"]
    data, sc = s["w"]
    if c["fmt"] == "q4":
        abi.call("mllm_gemv_q4", m, n, _p(data), _p(sc), GROUP, _p(s["x"]), _p(s["y"]), st)
    elif c["fmt"] == "f32":
        abi.call("mllm_gemv_f32", m, n, _p(data), _p(s["x"]), _p(s["y"]), st)
    else:
        abi.call("mllm_gemv_" + ("q8" if c["fmt"] == "q8" else "q8_g32"), m, n, _p(data), _p(sc), _p(s["x"]), _p(s["y"]), st)
    return s["y"]


# ---------------------------------------------------------------- work
def _mat_bytes(rows, cols, kind, group=GROUP):
    return {"q4": rows * cols // 2 + 4 * rows * (cols // group), "q8": rows * cols + 4 * rows,
            "q8g32": rows * cols + 4 * rows * (cols // 32), "f16": 2 * rows * cols, "bf16": 2 * rows * cols,
            "f32": 4 * rows * cols}[kind]


def work(case):
    c = case
    op = c["op"]
    if op == "mlp_ops":
        T, D, FF = c["tokens"], c["d_model"], c["d_ff"]
        b = 2 * _mat_bytes(FF, D, "q4") + _mat_bytes(D, FF, "q4") + 4 * D + 4 * T * (3 * D + FF)
        return {"bytes": b, "flops": 6 * T * D * FF}
    if op in ("argmax", "gemv", "stack", "dequant"):
        m, n, k = c["rows"], c["cols"], c.get("count", 1)
        out = m * n if op == "dequant" else m
        inp = 0 if op == "dequant" else n
        return {"bytes": k * (_mat_bytes(m, n, c.get("fmt", "q4")) + 4 * (inp + out)),
                "flops": m * n if op == "dequant" else 2 * k * m * n}
    D, FF, V, L, kvd = c["d_model"], c["d_ff"], c["vocab"], c["layers"], 64 * c["kv_heads"]
    up = 1 if c["arch"] == "gpt2" else 2
    shapes = [(D + 2 * kvd, D), (D, D)] + [(FF, D)] * up + [(D, FF)]
    layer = sum(_mat_bytes(r, k, c["kind"], c["group"]) for r, k in shapes)
    head = _mat_bytes(V, D, c["kind"], c["group"])
    params = sum(r * k for r, k in shapes)
    kvb = 2 if c["kv_fp16"] else 4
    # passes over the weights, tokens, rows of logits, first position
    if op == "prompt":
        passes, T, rows, p0 = 1, c["tokens"], 1, 0
    elif op == "verify":
        passes, T, rows, p0 = 1, c["steps"], c["steps"], c["ctx"]
    else:
        n = c["steps"] + (1 if op == "chain" else 0)
        passes, T, rows, p0 = n, n, n, c["ctx"]
    keys = sum(p0 + t + 1 for t in range(T))
    read = keys if passes > 1 else p0
    return {"bytes": passes * (L * layer + head) + 2 * kvd * kvb * L * (read + T) + 4 * rows * V,
            "flops": 2 * T * L * params + 2 * rows * V * D + 4 * D * L * keys}


# ---------------------------------------------------------------- tolerance
def tolerance(case):
    """About four times what the float32 kernels differ from 64 bits by on the
    listed and drawn cases: operators 1.2e-7 to 3e-7, whole models 3e-7 to
    4e-7 with the f32 cache and 7e-6 to 2.6e-5 with the f16 cache, where a
    value may round the other way."""
    op = case["op"]
    if op == "dequant":
        return "exact"
    if op in ("mlp_ops", "argmax", "gemv", "stack"):
        return {"rel": 1.2e-6, "max": 2e-5}
    return {"rel": 1e-4, "max": 1e-3} if case["kv_fp16"] else {"rel": 2e-6, "max": 3e-5}


# ---------------------------------------------------------------- 64 bits
class _Exact:
    """The model of infer.js in 64 bits (weights and tables as stored)."""

    def __init__(self, c, seed):
        self.c = c
        self.w = {n: (_plain(d, sc, st, c["group"]) if st != "f32" else d.double())
                  for n, d, sc, st in _tensors(c, seed)}
        self.quant = c["kind"] in ("q4", "q8", "q8g32")
        self.k = [None] * c["layers"]
        self.v = [None] * c["layers"]
        self.pos = 0
        inv = torch.tensor([1.0 / 100000.0 ** (2.0 * i / 64) for i in range(32)], dtype=torch.float64).float().double()
        ang = torch.arange(c["max_seq"], dtype=torch.float64)[:, None] * inv[None, :]
        self.cos = torch.cat([ang.cos(), ang.cos()], 1).float().double().to(DEV)
        self.sin = torch.cat([ang.sin(), ang.sin()], 1).float().double().to(DEV)

    def norm(self, x, name):
        w, D = self.w[name], self.c["d_model"]
        if self.c["arch"] == "gpt2":
            d = x - x.mean(-1, keepdim=True)
            return d / torch.sqrt((d * d).mean(-1, keepdim=True) + 1e-5) * w[:D] + w[D:]
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w

    def rope(self, x, p0):
        n = x.shape[1]
        rot = torch.cat([-x[..., 32:], x[..., :32]], -1)
        return x * self.cos[p0:p0 + n] + rot * self.sin[p0:p0 + n]

    def cached(self, x):
        return x.float().half().double() if self.c["kv_fp16"] else x

    def forward(self, ids):
        """The logits of every position of ids; the cache grows by them."""
        c, w = self.c, self.w
        D, NH, NKV, T, p0 = c["d_model"], c["heads"], c["kv_heads"], len(ids), self.pos
        gpt2 = c["arch"] == "gpt2"
        x = w["lm_head"][torch.tensor(ids, device=DEV)]
        if gpt2:
            x = (x / w["scale_factors"] if self.quant else x) + w["wpe"][p0:p0 + T]
        for i in range(c["layers"]):
            b = "blocks.%d." % i
            y = self.norm(x, b + ("ln1" if gpt2 else "norm1")) @ w[b + "attn.qkv"].T
            if gpt2:
                y = y + w[b + "attn.qkv_bias"]
            q = y[:, :D].reshape(T, NH, 64).transpose(0, 1)
            k = y[:, D:D + 64 * NKV].reshape(T, NKV, 64).transpose(0, 1)
            v = y[:, D + 64 * NKV:].reshape(T, NKV, 64).transpose(0, 1)
            if not gpt2:
                q, k = self.rope(q, p0), self.rope(k, p0)
            k, v = self.cached(k), self.cached(v)
            k = k if p0 == 0 else torch.cat([self.k[i], k], 1)
            v = v if p0 == 0 else torch.cat([self.v[i], v], 1)
            self.k[i], self.v[i] = k, v
            mask = torch.arange(p0 + T, device=DEV)[None, :] > torch.arange(p0, p0 + T, device=DEV)[:, None]
            o = []
            for h in range(NH):
                sc = (q[h] @ k[h * NKV // NH].T.contiguous()) / 8.0
                o.append(torch.softmax(sc.masked_fill(mask, -math.inf), -1) @ v[h * NKV // NH])
            o = torch.cat(o, 1) @ w[b + "attn.proj"].T
            x = x + (o + w[b + "attn.proj_bias"] if gpt2 else o)
            y = self.norm(x, b + ("ln2" if gpt2 else "norm2"))
            if gpt2:
                h = y @ w[b + "mlp.fc"].T + w[b + "mlp.fc_bias"]
                h = 0.5 * h * (1.0 + torch.tanh(0.7978845608028654 * (h + 0.044715 * h ** 3)))
                x = x + (h @ w[b + "mlp.proj"].T + w[b + "mlp.proj_bias"])
            else:
                h = torch.nn.functional.silu(y @ w[b + "mlp.w1"].T) * (y @ w[b + "mlp.w3"].T)
                x = x + h @ w[b + "mlp.w2"].T
        self.pos = p0 + T
        self.x = self.norm(x, "ln_f" if gpt2 else "norm_f")

    def logits(self, rows=slice(None)):
        return self.x[rows] @ self.w["lm_head"].T


def exact(case, seed):
    c = case
    op = c["op"]
    if op in ("chain", "prompt", "verify", "step"):
        m = _Exact(c, seed)
        ids, more = _ids(c, seed)
        m.forward(ids)
        if op == "prompt":
            return m.logits(-1)
        if op == "chain":
            tok, out = more[0], []
            for _ in range(c["steps"]):
                m.forward([tok])
                tok = int(m.logits(-1).argmax())
                out.append(tok)
            m.forward([tok])
            return {"ids": np.asarray(out, np.int64), "logits": m.logits(-1)}
        m.forward(more)
        lg = m.logits()
        return {"ids": lg.argmax(-1), "logits": lg} if op == "verify" else lg
    s = _op_inputs(c, seed)
    if op == "mlp_ops":
        x = s["x"].double()
        n = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * s["gain"].double()
        h = torch.nn.functional.silu(n @ _plain(*s["w1"], "q4").T) * (n @ _plain(*s["w3"], "q4").T)
        return {"n": n, "h": h, "y": h @ _plain(*s["w2"], "q4").T}
    if op == "stack":
        return [_plain(*w, c["fmt"]) @ x.double() for w, x in zip(s["w"], s["x"])]
    w = _plain(*s["w"], c.get("fmt", "q4"))
    if op == "dequant":
        return w
    y = w @ s["x"].double()
    return {"y": y, "id": y.argmax().reshape(1)} if op == "argmax" else y
