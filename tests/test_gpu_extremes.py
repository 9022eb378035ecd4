"""The kind-generic models on values at the ends of float32's and f16's ranges:
what one call leaves in the KV cache or computes for one token must not reach
results that do not depend on it."""
import dataclasses

import numpy as np
import pytest

import mllm
from mllm import pgw

gpu = pytest.mark.gpu
A, B = 5, 9  # tokens: only A's embedding has component 0


def bits(a):
    return np.array(a, np.float32).view(np.uint32)


def edited(arch, edit, seed=61, **kw):
    """An f32 model whose matrices edit(w) changes in place; w(name): a matrix."""
    model = {k: kw.pop(k) for k in ("bias_std", "std") if k in kw}
    b = pgw.parse_pgw(pgw.make_model(pgw.small_config(arch, **kw), seed=seed, kind="f32", **model))
    buf = bytearray(b.buffer)

    def w(name):
        t = b.tensors[name]
        n = int(np.prod(t["shape"]))
        return np.frombuffer(buf, np.float32, n, b.payload_off + t["offset"]).reshape(t["shape"])

    edit(w)
    return dataclasses.replace(b, buffer=bytes(buf))


@gpu
@pytest.mark.parametrize("kv_fp16", [False, True])
@pytest.mark.parametrize("calls", ["prompt 1", "prompt 2", "verify"])
def test_first_position_ignores_the_old_cache(calls, kv_fp16):
    """Token A leaves an infinite value row (and NaN in the deeper layers) at
    position 0.  Calls that start there again give a fresh model's bits."""
    def edit(w):
        w("lm_head")[:, 0] = 0.0
        w("lm_head")[A, 0] = 1.0
        v = w("blocks.0.attn.qkv")
        v[192 + 64:, 0] = 3e38  # value rows: infinite for A, untouched for the others

    bundle = edited("llama", edit, d_model=192, n_heads=3, n_kv_heads=1)
    print(f"old cache {calls} fp16={kv_fp16}", flush=True)

    def results(g):
        if calls == "verify":
            g.cacheLen = 0
            return g.forwardVerify([B, 11, 12], want_logits=True)[1]
        first = g.forwardPrompt([B] if calls == "prompt 1" else [B, 11]).copy()
        return np.stack([first, g.forwardDecode(13).copy()])

    fresh, used = (mllm.PetitGPT(bundle, kv_fp16=kv_fp16) for _ in range(2))
    want = results(fresh)
    assert np.isfinite(want).all()
    assert not np.isfinite(used.forwardPrompt([A])).any()
    assert np.array_equal(bits(results(used)), bits(want))
    fresh.destroy()
    used.destroy()


def rel(a, b):
    return float(np.abs(a - b).max()) / float(np.abs(b).max())


@gpu
@pytest.mark.parametrize("n", [32, 256, 1024])
@pytest.mark.parametrize("how", ["step", "prompt"])
def test_minus_infinite_scores_weigh_nothing(oracle_lib, how, n):
    """The keys 0 .. n-1 are infinite in an f16 cache and score -inf for the last
    token, whose own key is finite and alone in its 32 positions (n = 256: in its
    256, n = 1024: in the fifth split).  They get weight 0, as in the oracle,
    where the same scores are about -1e6."""
    def edit(w):
        w("lm_head")[:, 0] = 0.0
        w("lm_head")[A, 0] = w("lm_head")[B, 0] = 1.0  # B too, so that its query has component 31
        w("lm_head")[:, 1] = 0.0
        w("lm_head")[A, 1] = 1.0
        qkv = w("blocks.0.attn.qkv")
        qkv[[31, 128 + 31]] = 0.0  # component 31 turns by less than 0.2 over 1100 positions
        qkv[31, 0] = -1.0
        qkv[128 + 31, 1] = 1e5     # A's keys only

    bundle = edited("llama", edit, n_layers=1, max_seq_len=1100)
    print(f"-inf scores {how} n={n}", flush=True)
    g = mllm.PetitGPT(bundle, kv_fp16=True)
    ref = oracle_lib.OracleModel(bundle)
    if how == "step":
        g.forwardPrompt([A] * n)
        got = g.forwardDecode(B).copy()
    else:
        got = g.forwardPrompt([A] * n + [B]).copy()
    want = ref.forward_prompt([A] * n + [B])
    g.destroy()
    ref.close()
    assert rel(got, want) <= 5e-3  # the f16 cache


@gpu
@pytest.mark.parametrize("arch", ["llama", "gpt2"])
@pytest.mark.parametrize("v,qk", [(-10, 0), (-30, 0), (17, 0), (60, 0), (0, -30), (0, 20), (0, 60), (-20, -20)])
def test_prompt_attention_at_any_magnitude(oracle_lib, arch, v, qk):
    """Value rows times 2^v with the output projection times 2^-v, query rows
    times 2^-qk with key rows times 2^qk: the same function.  Last logits of a
    batched prompt and of a step after it within 2e-6 of the float64 oracle's
    scale (float32 roundings, 2e-7 to 6e-7 measured)."""
    def edit(w):
        for i in range(2):
            q = w(f"blocks.{i}.attn.qkv")
            q[:128] *= 2.0 ** -qk
            q[128:-64 * kv] *= 2.0 ** qk
            q[-64 * kv:] *= 2.0 ** v
            w(f"blocks.{i}.attn.proj")[:] *= 2.0 ** -v

    kv = 1 if arch == "llama" else 2
    bundle = edited(arch, edit, max_seq_len=160)
    ids = [int(t) for t in np.random.default_rng(62).integers(0, 512, 101)]
    print(f"magnitude {arch} v=2^{v} qk=2^{qk}", flush=True)
    g = mllm.PetitGPT(bundle)
    ref = oracle_lib.OracleModel(bundle)
    w = [rel(g.forwardPrompt(ids[:100]), ref.forward_prompt(ids[:100])),
         rel(g.forwardDecode(ids[100]), ref.forward_decode(ids[100]))]
    g.destroy()
    ref.close()
    assert max(w) <= 2e-6, w


@gpu
@pytest.mark.parametrize("kv_fp16", [False, True])
@pytest.mark.parametrize("at", [21, 60])
def test_infinite_value_stays_with_later_tokens(at, kv_fp16):
    """Token A's value row is infinite.  The cache rows of the prompt's tokens
    before it serve a step after a roll-back as those of a prompt without it do
    (to 2e-6 of the logits' scale: the products' split over waves may differ;
    f16 cache: a rounding the other way)."""
    def edit(w):
        w("lm_head")[:, 0] = 0.0
        w("lm_head")[A, 0] = 1.0
        w("blocks.0.attn.qkv")[128 + 64:, 0] = 3e38

    bundle = edited("llama", edit, max_seq_len=128)
    ids = [int(t) for t in np.random.default_rng(63).integers(10, 512, 90)]
    print(f"infinite value at {at} fp16={kv_fp16}", flush=True)
    g = mllm.PetitGPT(bundle, kv_fp16=kv_fp16)
    g.forwardPrompt(ids[:at])
    want = g.forwardDecode(B).copy()
    assert not np.isfinite(g.forwardPrompt(ids[:at] + [A] + ids[at:])).any()
    g.cacheLen = at
    got = g.forwardDecode(B).copy()
    g.destroy()
    assert rel(got, want) <= (5e-3 if kv_fp16 else 2e-6)


@gpu
@pytest.mark.parametrize("kind", ["f32", "f16", "bf16", "q8"])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("name", ["attn.qkv", "attn.proj", "mlp.w1", "mlp.w3", "mlp.w2"])
def test_prompt_shows_non_finite_weights(name, value, kind):
    """One infinite or NaN weight (q8: row scale) of layer 0 leaves no finite
    logit in a batched prompt, as in the token steps."""
    b = pgw.parse_pgw(pgw.make_model(pgw.small_config(), seed=64, kind=kind))
    buf = bytearray(b.buffer)
    t = b.tensors["blocks.0." + name]
    row = -1 if name == "attn.qkv" else 7  # a value row
    if kind == "q8":
        np.frombuffer(buf, np.float32, t["shape"][0], b.payload_off + t["scaleOffset"])[row] = value
    else:
        bits16 = {"f16": int(np.float16(value).view(np.uint16)), "bf16": int(np.float32(value).view(np.uint32)) >> 16}
        dt = np.float32 if kind == "f32" else np.uint16
        m = np.frombuffer(buf, dt, int(np.prod(t["shape"])), b.payload_off + t["offset"]).reshape(t["shape"])
        m[row, 3] = value if kind == "f32" else bits16[kind]
    g = mllm.PetitGPT(dataclasses.replace(b, buffer=bytes(buf)))
    print(f"weight {name} {kind} {value}", flush=True)
    batch = g.forwardPrompt([3, 1, 4, 1, 5]).copy()
    steps = [g.forwardPrompt([3, 1])] + [g.forwardDecode(t) for t in (4, 1, 5)]
    assert not np.isfinite(steps[-1]).any()
    assert not np.isfinite(batch).any()
    g.destroy()
