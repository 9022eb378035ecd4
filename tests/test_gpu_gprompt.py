"""Batched prompts of the kind-generic models (mllm_gprompt.hip; forwardPrompt,
infer.js:553-577) against the oracle, which accumulates in float64: every
storage at lengths around the 32-token tile, the workgroup order by XCD (one to
eight token groups of XCDs), a chunk boundary, partial rotary, four
query heads per KV head, gate and up rows in different storages.

Bar: the last-token logits, and those of decode steps that read the cache,
within TOL of the oracle relative to their scale: the GEMMs' operands are
exact (Q8 group-32 and Q4 weights rounded once to float32), so what is left
are float32 roundings, 2e-7 to 5e-7 measured, as in the token steps.
"""
import numpy as np
import pytest

import mllm
from mllm import pgw

gpu = pytest.mark.gpu
TOL = 2e-6
TOL_F16KV = 5e-3  # K or V elements may round to neighbouring f16 values


def build(arch="llama", seed=1, std=0.02, **kw):
    model = {k: kw.pop(k) for k in ("kind", "group", "storages", "bias_std") if k in kw}
    return pgw.parse_pgw(pgw.make_model(pgw.small_config(arch, **kw), seed=seed, std=std, **model))


def worst(oracle_lib, bundle, n, kv_fp16=False):
    g = mllm.PetitGPT(bundle, kv_fp16=kv_fp16)
    assert g.decodeKernel == "generic kernels"
    ref = oracle_lib.OracleModel(bundle)
    ids = [int(v) for v in np.random.default_rng(n).integers(0, bundle.cfg.vocab_size, n + 2)]
    rows = [(g.forwardPrompt(ids[:n]).copy(), ref.forward_prompt(ids[:n]))]
    rows += [(g.forwardDecode(t).copy(), ref.forward_decode(t)) for t in ids[n:]]
    assert g.cacheLen == n + 2
    g.destroy()
    ref.close()
    return max(float(np.abs(a - b).max()) / float(np.abs(b).max()) for a, b in rows)


@gpu
@pytest.mark.parametrize("arch", ["llama", "gpt2"])
@pytest.mark.parametrize("kind,group", [("f32", 32), ("f16", 32), ("bf16", 32), ("q8", 32), ("q8g32", 32), ("q4", 64),
                                        ("q4", 8)])
@pytest.mark.parametrize("n", [3, 32, 33, 100])
def test_kind_prompt_vs_oracle(oracle_lib, arch, kind, group, n):
    extra = {"bias_std": 0.02} if arch == "gpt2" else {}
    bundle = build(arch, seed=41, kind=kind, group=group, d_model=192, n_heads=3, d_ff=320, max_seq_len=160,
                   n_kv_heads=3 if arch == "gpt2" else 1, **extra)
    print(f"prompt {arch} {kind}/{group} n={n}", flush=True)
    assert worst(oracle_lib, bundle, n) <= TOL


def token_groups(n, rows, planes):
    """The token groups of XCDs that a GEMM of n tokens takes: the split whose
    XCDs fetch least, in bytes per column."""
    w, x = rows * 2 * planes, (n + 31) // 32 * 32 * 6
    return min((1, 2, 4, 8), key=lambda t: t * w + 8 // t * x)


def test_tile_placement_reaches_every_split():
    rows = (256 + 2 * 64, 256, 512)  # QKV, O and down, gate/up
    assert {token_groups(n, r, 1) for n in (20, 100, 300, 512) for r in rows} == {1, 2, 4, 8}


@gpu
@pytest.mark.parametrize("n", [20, 100, 255, 256, 300, 512])
def test_tile_placement_vs_oracle(oracle_lib, n):
    """XCDs in one to eight token groups, and tile counts that do and do not
    divide among them."""
    bundle = build(seed=42, kind="bf16", d_model=256, n_heads=4, n_kv_heads=1, max_seq_len=640)
    print(f"placement n={n}", flush=True)
    assert worst(oracle_lib, bundle, n) <= TOL


@gpu
@pytest.mark.parametrize("kv_fp16", [False, True])
@pytest.mark.parametrize("n", [33, 448, 449])
def test_attention_halves_vs_oracle(oracle_lib, n, kv_fp16):
    """Nine heads: 18, 126 and 135 (tile, head) workgroups, the output's halves
    apart up to 128; up to 15 key blocks on eight waves."""
    bundle = build(seed=49, kind="bf16", n_layers=1, d_model=576, n_heads=9, n_kv_heads=3, max_seq_len=512)
    print(f"halves n={n} fp16={kv_fp16}", flush=True)
    assert worst(oracle_lib, bundle, n, kv_fp16) <= (TOL_F16KV if kv_fp16 else TOL)


@gpu
@pytest.mark.parametrize("n", [2048, 2049, 2085])
def test_chunk_boundary_vs_oracle(oracle_lib, n):
    """More tokens than a chunk holds: the second chunk reads the first's keys."""
    bundle = build(seed=43, kind="q8", n_layers=1, max_seq_len=2100)
    print(f"chunk n={n}", flush=True)
    assert worst(oracle_lib, bundle, n) <= TOL


@gpu
@pytest.mark.parametrize("case", ["partial rotary", "mixed gate/up", "f16 cache", "q4 large d_ff"])
def test_prompt_options_vs_oracle(oracle_lib, case):
    print(case, flush=True)
    if case == "partial rotary":
        assert worst(oracle_lib, build(seed=44, kind="f16", rope_pct=0.5), 50) <= TOL
    elif case == "mixed gate/up":
        for a, b in (("q8", "f32"), ("f16", "bf16"), ("q4", "q8")):
            st = {"blocks.0.mlp.w1": a, "blocks.0.mlp.w3": b, "blocks.1.attn.qkv": "f16"}
            assert worst(oracle_lib, build(seed=45, kind="bf16", storages=st), 40) <= TOL
    elif case == "f16 cache":
        assert worst(oracle_lib, build(seed=46, kind="f32", n_layers=1), 60, kv_fp16=True) <= TOL_F16KV
    else:  # Q4 group-32 beyond the fused step's limits
        assert worst(oracle_lib, build(seed=47, kind="q4", d_ff=4160, n_layers=1), 45) <= TOL


@gpu
@pytest.mark.parametrize("n", [1, 3, 40])
@pytest.mark.parametrize("kind", ["f16", "q4"])
def test_set_prefill_0_gives_the_token_steps(kind, n):
    """Batches switched off: the token steps' bits, the bytes of the bf16 copy
    given back, and thresholds refused as before."""
    bundle = build(seed=48, kind=kind, group=64)
    ids = [int(v) for v in np.random.default_rng(n).integers(0, 512, n + 1)]
    print(f"set_prefill 0 {kind} n={n}", flush=True)
    g = mllm.PetitGPT(bundle)
    steps = g.forwardPrompt(ids[:1]).copy()
    for t in ids[1:n]:
        steps = g.forwardDecode(t).copy()
    before = g.bytesAllocated
    for _ in range(2):  # a second time changes nothing
        g.set_prefill(0)
        c = bundle.cfg
        weights = c.n_layers * c.d_model * (2 * c.d_model + 2 * 64 * c.n_kv_heads + 3 * c.d_ff)
        assert before - g.bytesAllocated >= weights * (4 if kind == "f16" else 6)
        got = g.forwardPrompt(ids[:n]).copy()
        assert g.cacheLen == n and np.array_equal(got.view(np.uint32), steps.view(np.uint32))
        with pytest.raises(mllm.abi.MllmError, match="UNSUPPORTED"):
            g.set_prefill(3)
    g.destroy()
