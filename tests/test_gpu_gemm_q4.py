"""mllm_gemm_q4 on the matrix cores: every row carries the bits of
mllm_gemv_q4 on that token, at the edges of the 32-token, 32-row and staging
tiles and for every form of the summation order (groups per lane 1 .. 8, one
lane .. 64)."""
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
