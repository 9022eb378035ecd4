"""The kind-generic decode step's kernels at the edges of their splits: rows
that fit a lane's registers and longer ones, segments of every length, the
attention's 32-position waves and 256-position workgroups, more splits than are
merged at once.  Bar: within TOL of the float64 oracle, relative to the
logits' scale (float32 roundings: 2e-7 to 6e-7 measured)."""
import numpy as np
import pytest

import mllm
from mllm import pgw

gpu = pytest.mark.gpu
TOL = 2e-6
TOL_F16KV = 5e-3


def build(arch, seed, **kw):
    model = {k: kw.pop(k) for k in ("kind", "group", "storages", "bias_std") if k in kw}
    return pgw.parse_pgw(pgw.make_model(pgw.small_config(arch, **kw), seed=seed, **model))


def rel(a, b):
    return float(np.abs(a - b).max()) / float(np.abs(b).max())


@gpu
@pytest.mark.parametrize("kv_fp16", [False, True])
@pytest.mark.parametrize("n", [1, 31, 32, 254, 256, 1023, 1290])
def test_attention_splits_vs_oracle(oracle_lib, n, kv_fp16):
    """Decode at positions on both sides of a wave, a workgroup and four
    workgroups; three query heads per KV head."""
    bundle = build("llama", 51, kind="f16", n_layers=1, d_model=192, n_heads=3, n_kv_heads=1, max_seq_len=1300)
    g = mllm.PetitGPT(bundle, kv_fp16=kv_fp16)
    ref = oracle_lib.OracleModel(bundle)
    ids = [int(v) for v in np.random.default_rng(n).integers(0, bundle.cfg.vocab_size, n + 3)]
    print(f"attention n={n} fp16={kv_fp16}", flush=True)
    g.forwardPrompt(ids[:n])
    ref.forward_prompt(ids[:n])
    w = max(rel(g.forwardDecode(t), ref.forward_decode(t)) for t in ids[n:])
    g.destroy()
    ref.close()
    assert w <= (TOL_F16KV if kv_fp16 else TOL), w


@gpu
@pytest.mark.parametrize("kind", ["f32", "f16", "q8", "q8g32", "q4"])
@pytest.mark.parametrize("arch,d_model,d_ff", [("llama", 64, 64), ("llama", 576, 1536), ("gpt2", 768, 704),
                                               ("llama", 2112, 4160), ("gpt2", 2112, 320)])
def test_rows_vs_oracle(oracle_lib, kind, arch, d_model, d_ff):
    """Rows of 64 to 4160 columns: the last shapes are past a lane's registers
    in f32 (2112) and in every storage (4160)."""
    h = d_model // 64
    bundle = build(arch, 52, kind=kind, group=64, n_layers=1, vocab_size=100, d_model=d_model, n_heads=h,
                   n_kv_heads=h if arch == "gpt2" or h % 3 else h // 3, d_ff=d_ff, max_seq_len=16,
                   **({"bias_std": 0.02} if arch == "gpt2" else {}))
    g = mllm.PetitGPT(bundle)
    assert g.decodeKernel == "generic kernels"
    ref = oracle_lib.OracleModel(bundle)
    print(f"rows {arch} {kind} {d_model}x{d_ff}", flush=True)
    w = [rel(g.forwardPrompt([3, 5]), ref.forward_prompt([3, 5]))]  # two tokens: the token steps
    w += [rel(g.forwardDecode(t), ref.forward_decode(t)) for t in (7, 11)]
    x = np.random.default_rng(1).standard_normal(d_ff).astype(np.float32)
    name = "blocks.0.mlp.proj" if arch == "gpt2" else "blocks.0.mlp.w2"
    w.append(rel(g.gemv(name, x), ref.gemv(name, x)))
    g.destroy()
    ref.close()
    assert max(w) <= TOL, w


@gpu
@pytest.mark.parametrize("vocab", [5, 8191, 8192, 17001])
def test_argmax_vs_logits(vocab):
    """Vocabularies around the argmax's 8192 loads at a time."""
    g = mllm.PetitGPT(build("llama", 53, kind="bf16", n_layers=1, vocab_size=vocab))
    print(f"argmax vocab={vocab}", flush=True)
    for t in range(4):
        lg = g.forwardPrompt([t, 1]) if t == 0 else g.forwardDecode(t)
        assert g.last_argmax == int(np.argmax(lg))
    g.destroy()


@gpu
@pytest.mark.parametrize("kind", ["f32", "f16", "q8", "q8g32", "q4"])
@pytest.mark.parametrize("arch,kv_fp16", [("llama", False), ("llama", True), ("gpt2", False)])
def test_verify_pass_rows_bit_identical_to_decode(arch, kv_fp16, kind):
    """A pass of 2, 7 and 16 tokens over an attention split's edge, rows in and
    past a lane's registers: logits, argmax and the cache it leaves (read by the
    next decode) as single steps give them, bit for bit."""
    h = 6
    bundle = build(arch, 54, kind=kind, group=64, n_layers=2, vocab_size=700, d_model=64 * h, n_heads=h,
                   n_kv_heads=h if arch == "gpt2" else 2, d_ff=4160, max_seq_len=300,
                   **({"bias_std": 0.02} if arch == "gpt2" else {}))
    g = mllm.PetitGPT(bundle, kv_fp16=kv_fp16)
    ids = [int(v) for v in np.random.default_rng(55).integers(0, 700, 280)]
    print(f"verify {arch} {kind} fp16={kv_fp16}", flush=True)
    for n, m in ((2, 2), (30, 7), (250, 16)):
        g.forwardPrompt(ids[:n])
        am, lg = g.forwardVerify(ids[n:n + m], want_logits=True)
        after = g.forwardDecode(ids[n + m]).copy()
        g.cacheLen = n
        for i in range(m):
            row = g.forwardDecode(ids[n + i])
            assert np.array_equal(row.view(np.uint32), lg[i].view(np.uint32)), (n, m, i)
            assert am[i] == g.last_argmax
        assert np.array_equal(after.view(np.uint32), g.forwardDecode(ids[n + m]).view(np.uint32))
    g.destroy()


@gpu
@pytest.mark.parametrize("kind", ["q4", "q8"])
@pytest.mark.parametrize("vocab", [64, 641])
def test_outputs_of_every_call_shape(kind, vocab):
    """Both engines' outputs at the host: 1 to 16 rows, with and without the
    logits or the argmax, after larger calls and chains of every short length."""
    import ctypes as C
    from mllm import abi
    g = mllm.PetitGPT(build("llama", 57, kind=kind, n_layers=2, vocab_size=vocab, max_seq_len=64))
    ids = [int(v) for v in np.random.default_rng(58).integers(0, vocab, 64)]
    print(f"outputs {kind} V={vocab}", flush=True)
    rows = np.empty((40, vocab), np.float32)
    g.forwardPrompt(ids[:4])
    for i in range(40):
        rows[i] = g.forwardDecode(ids[4 + i])
        assert g.last_argmax == int(rows[i].argmax())
    for m in (16, 1, 2, 15, 3):
        g.cacheLen = 4
        am, lg = g.forwardVerify(ids[4:4 + m], want_logits=True)
        assert np.array_equal(lg.view(np.uint32), rows[:m].view(np.uint32)) and am == [int(v) for v in rows[:m].argmax(1)]
        g.cacheLen = 4
        assert g.forwardVerify(ids[4:4 + m])[0] == am
    a = np.array(ids[:5], np.int32)
    for call, lead in (("mllm_forward_decode", (ids[4],)), ("mllm_forward_prompt", (a.ctypes.data, 5))):
        out, am = np.zeros(vocab, np.float32), C.c_int32(-1)
        for lp, ap in ((out.ctypes.data, None), (None, C.byref(am)), (None, None)):
            g.cacheLen = 4
            abi.call(call, g._h, *lead, lp, ap)
            assert g.cacheLen == 5
        assert am.value == int(out.argmax())
    g.cacheLen = 4
    chain = g.decodeChain(ids[4], 20)
    for n in (1, 7, 19):
        g.cacheLen = 4
        assert g.decodeChain(ids[4], n) == chain[:n]
    g.destroy()
