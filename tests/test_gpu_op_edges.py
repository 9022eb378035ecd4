"""Operators at the edges of their launch rules.  mllm_gemm_q4 on the matrix
cores: every row carries the bits of mllm_gemv_q4 on that token, at the edges
of the 32-token, 32-row and staging tiles and for every form of the summation
order (groups per lane 1 .. 8, one lane .. 64).  mllm_dequant_q4 at every
alignment, mllm_gemv_f32 with one and with four rows per wave."""
import ctypes as C

import numpy as np
import pytest

from mllm import abi, pgw

torch = pytest.importorskip("torch")
gpu = pytest.mark.gpu


def ptr(t):
    return C.c_void_p(t.data_ptr())


def check(t, m, n, x):
    rng = np.random.default_rng(t * 7 + m * 3 + n)
    packed, sc = pgw.quant_q4((rng.standard_normal((m, n)) * 0.02).astype(np.float32))
    dp, ds, dx = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (packed, sc, x))
    y = torch.full((t + 1, m), 7.0, dtype=torch.float32, device="cuda")
    one = torch.empty((t, m), dtype=torch.float32, device="cuda")
    abi.call("mllm_gemm_q4", t, m, n, ptr(dp), ptr(ds), 32, ptr(dx), ptr(y), None)
    for i in range(t):
        abi.call("mllm_gemv_q4", m, n, ptr(dp), ptr(ds), 32, ptr(dx[i]), ptr(one[i]), None)
    torch.cuda.synchronize()
    got, want = y.cpu().numpy(), one.cpu().numpy()
    assert (got[t] == 7.0).all()  # nothing past the last token
    same = (got[:t].view(np.uint32) == want.view(np.uint32)) | (np.isnan(got[:t]) & np.isnan(want))
    assert same.all(), (t, m, n, int((~same).sum()))


@gpu
@pytest.mark.parametrize("t", [31, 32, 33, 77])
@pytest.mark.parametrize("m,n", [(1, 32), (31, 64), (33, 96), (320, 576), (257, 960), (300, 1536), (129, 2560),
                                 (64, 4960), (40, 8192), (33, 16384)])
def test_rows_bit_identical_to_gemv(t, m, n):
    print(f"gemm t={t} m={m} n={n}", flush=True)
    check(t, m, n, np.random.default_rng(t + n).standard_normal((t, n)).astype(np.float32))


@gpu
@pytest.mark.parametrize("t", [47, 48, 49])
@pytest.mark.parametrize("m,n", [(33, 4096), (40, 4128), (33, 8192), (33, 12288)])
def test_tokens_where_the_matrix_cores_take_over(t, m, n):
    """Rows on more than 16 lanes change over at 48 tokens."""
    print(f"gemm t={t} m={m} n={n}", flush=True)
    check(t, m, n, np.random.default_rng(t + n).standard_normal((t, n)).astype(np.float32))


@gpu
@pytest.mark.parametrize("t,m,n", [(1000, 2300, 960), (1030, 2050, 2560), (520, 4100, 544), (530, 4100, 4096)])
def test_large_launches(t, m, n):
    """A workgroup of eight waves per CU: fewer groups fit the LDS at a time."""
    print(f"gemm t={t} m={m} n={n}", flush=True)
    check(t, m, n, np.random.default_rng(1).standard_normal((t, n)).astype(np.float32))


@gpu
def test_values_over_the_range():
    """Zero groups, groups of one value, magnitudes from 1e-30 to 1e30 in a
    row, infinities and NaN: the same bits (NaN where the GEMV has NaN)."""
    rng = np.random.default_rng(2)
    t, n = 40, 320
    x = rng.standard_normal((t, n)).astype(np.float32)
    x[0] = 0
    x[1, 32:64] = 0
    x[2, :] = 0
    x[2, 5] = 3.5
    x[3] *= np.float32(10.0) ** rng.integers(-30, 30, n).astype(np.float32)
    x[4] = -x[4].max()
    x[5, 7] = np.inf
    x[6, 8] = np.nan
    x[7, 40:50] = -np.inf
    check(t, 100, n, x)


@gpu
def test_gemm_groups_below_the_scaled_range():
    """Groups whose largest value is below 2.3e-32, where the GEMV's scale
    overflows and its integers wrap: still the GEMV's bits."""
    rng = np.random.default_rng(3)
    t, n = 40, 320
    x = rng.standard_normal((t, n)).astype(np.float32)
    x[::2, 32:64] *= np.float32(1e-33)
    x[1::2, 64:128] *= np.float32(1e-38)
    x[3] *= np.float32(1e-36)
    print("gemm tiny groups", flush=True)
    check(t, 100, n, x)


@gpu
@pytest.mark.parametrize("m,n", [(1, 32), (3, 96), (127, 160), (33, 4096), (2049, 4096)])
@pytest.mark.parametrize("skip", [0, 1, 2])
def test_dequant_every_alignment(m, n, skip):
    """Exact at sizes around a workgroup's 1024 quads, from packed bytes at any
    address into 16- and 8-byte aligned floats, nothing written past the end."""
    rng = np.random.default_rng(m + n)
    packed, sc = pgw.quant_q4(rng.standard_normal((m, n)).astype(np.float32))
    dp = torch.zeros(skip + packed.size, dtype=torch.uint8, device="cuda")
    dp[skip:] = torch.from_numpy(packed.reshape(-1).copy()).cuda()
    ds = torch.from_numpy(sc).cuda()
    out = torch.full((2 * skip + m * n + 4,), 7.0, dtype=torch.float32, device="cuda")
    print(f"dequant {m}x{n} skip={skip}", flush=True)
    abi.call("mllm_dequant_q4", m, n, C.c_void_p(dp.data_ptr() + skip), ptr(ds), 32,
             C.c_void_p(out.data_ptr() + 8 * skip), None)
    torch.cuda.synchronize()
    o = out.cpu().numpy()
    assert np.array_equal(o[2 * skip:2 * skip + m * n].reshape(m, n), pgw.dequant_q4(packed, sc))
    assert (o[:2 * skip] == 7.0).all() and (o[2 * skip + m * n:] == 7.0).all()


@gpu
@pytest.mark.parametrize("n", [1, 63, 64, 320, 577])
def test_gemv_f32_rows_per_wave(n):
    """The same rows with four rows per wave (16387 rows, the last wave short)
    and with one (their first 1000): the same bits, and within the float32 sum's
    bound of the float64 result."""
    rng = np.random.default_rng(n)
    m = 16387
    w, x = rng.standard_normal((m, n)).astype(np.float32), rng.standard_normal(n).astype(np.float32)
    dw, dx = torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda()
    y = torch.full((m + 1,), 7.0, dtype=torch.float32, device="cuda")
    y1 = torch.empty(1000, dtype=torch.float32, device="cuda")
    print(f"gemv f32 n={n}", flush=True)
    abi.call("mllm_gemv_f32", m, n, ptr(dw), ptr(dx), ptr(y), None)
    abi.call("mllm_gemv_f32", 1000, n, ptr(dw), ptr(dx), ptr(y1), None)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    assert got[m] == 7.0 and np.array_equal(got[:1000], y1.cpu().numpy())
    bound = (n + 8) * 2.0**-24 * (np.abs(w).astype(np.float64) @ np.abs(x).astype(np.float64))
    assert (np.abs(got[:m] - w.astype(np.float64) @ x.astype(np.float64)) <= bound).all()


@gpu
@pytest.mark.parametrize("m,n", [(19999, 576), (16387, 580), (16387, 673), (16387, 1024), (16386, 1025), (16387, 1028)])
def test_gemv_f32_rows_and_streams(m, n):
    """Four, two and one row per wave past 16384 rows, with ordinary and with
    streamed loads: the bits of a short call on the last rows (one row per wave,
    ordinary loads)."""
    rng = np.random.default_rng(m + n)
    w, x = torch.from_numpy(rng.random((m, n), np.float32) - 0.5).cuda(), torch.from_numpy(rng.random(n, np.float32)).cuda()
    y = torch.full((m + 1,), 7.0, dtype=torch.float32, device="cuda")
    k = 1000 + (m & 3)  # the tail starts on a 16-byte boundary
    y1 = torch.empty(k, dtype=torch.float32, device="cuda")
    print(f"gemv f32 {m}x{n}", flush=True)
    abi.call("mllm_gemv_f32", m, n, ptr(w), ptr(x), ptr(y), None)
    abi.call("mllm_gemv_f32", k, n, ptr(w[m - k:]), ptr(x), ptr(y1), None)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    assert got[m] == 7.0 and np.array_equal(got[m - k:m].view(np.uint32), y1.cpu().numpy().view(np.uint32))


@gpu
@pytest.mark.parametrize("rows", [57216, 57344, 57345])
@pytest.mark.parametrize("kind", ["first of ties", "nan0", "nan rows", "all nan"])
def test_argmax_on_both_sides_of_two_launches(rows, kind):
    """128 rows a tile: 447 tiles (one launch) and 448 or 449 (two), called
    twice on the same scratch, the index by infer.js:240-250."""
    rng = np.random.default_rng(rows)
    n = 64
    packed, sc = pgw.quant_q4(rng.standard_normal((rows, n)).astype(np.float32))
    x = rng.standard_normal(n).astype(np.float32)
    if kind == "first of ties":
        best = int(np.argmax(pgw.dequant_q4(packed, sc) @ x))
        packed[[rows - 1, rows // 2]] = packed[best]
        sc[[rows - 1, rows // 2]] = sc[best]
    elif kind == "nan0":
        sc[0, 0] = np.nan
    elif kind == "nan rows":
        sc[1::5, 1] = np.nan
    else:
        sc[:, 0] = np.nan
    dp, ds, dx = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (packed, sc, x))
    y = torch.empty(rows, dtype=torch.float32, device="cuda")
    i = torch.full((1,), -5, dtype=torch.int32, device="cuda")
    print(f"argmax rows={rows} {kind}", flush=True)
    for _ in range(2):
        i.fill_(-5)
        abi.call("mllm_gemv_q4_argmax", rows, n, ptr(dp), ptr(ds), 32, ptr(dx), ptr(y), ptr(i), None)
        torch.cuda.synchronize()
        v = y.cpu().numpy()
        want = 0 if np.isnan(v[0]) or np.isnan(v).all() else int(np.nanargmax(v))
        assert int(i.item()) == want
