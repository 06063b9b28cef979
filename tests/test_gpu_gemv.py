"""Dense layers on one to six rows, a wave per few columns (seven: the tile kernels), against fp64 products.  A sum of K products in any order
is off by at most K 2^-24 of the sum of magnitudes.  Here a lane adds K / 64 of them, six halvings and up to four parts follow, then bias,
residual and their sum: (K / 64 + 16) 2^-24 bounds it; the tile kernels' eight waves add K / 8 each in order, and four more."""
import zlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("n,k", [(1, 4), (3, 252), (16, 256), (33, 260), (70, 512), (5, 516), (2304, 768), (129, 1020), (40, 1024),
                                 (17, 1028), (7, 2048), (768, 3072), (50, 4092), (31, 4096), (30, 4100)])  # (the last: tile kernels)
def test_dense_rows_few(fdx, m, n, k):
    print("dense rows few", m, n, k, flush=True)
    assert fdx.lib.fdx_debug_dense_rows_form(m, n, k, 0) == (m <= 6 and k <= 4096)
    assert fdx.lib.fdx_debug_dense_rows_form(m, n, k, 1) == (m <= 6 and k <= 1024)
    steps = (k / 64 if m <= 6 and k <= 4096 else k / 8) + 16
    r = np.random.default_rng(zlib.crc32(repr((m, n, k)).encode()))
    x, w = r.standard_normal((m, k)).astype(np.float32), (r.standard_normal((n, k)) / np.sqrt(k)).astype(np.float32)
    b, res = r.standard_normal(n).astype(np.float32), r.standard_normal((m, n)).astype(np.float32)
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    size = np.abs(x64) @ np.abs(w64).T + np.abs(b) + np.abs(res)
    dx, dw, db, dr = (fdx.DevBuf.from_host(a) for a in (x, w, b, res))
    out = fdx.DevBuf(4 * m * n)
    relu = fdx.relu_act(1.5)
    fdx.check(fdx.lib.fdx_dense_rows_f32(fdx._dp(dx), m, k, fdx._dp(dw), fdx._dp(db), n, fdx._dp(dr), fdx.ctypes.byref(relu), fdx._dp(out)))
    got = out.to_host((m, n))
    want = np.clip(x64 @ w64.T + b + res, 0, 1.5)
    assert (np.abs(got - want) <= steps * EPS * size).all()
    fdx.check(fdx.lib.fdx_dense_rows_noalloc_f32(fdx._dp(dx), m, k, fdx._dp(dw), None, n, None, None, fdx._dp(out)))
    plain = out.to_host((m, n))
    assert (np.abs(plain - x64 @ w64.T) <= steps * EPS * size).all()
    if k > 1024:
        return
    wf, ws, bf = fdx.DevBuf(4 * n * k), fdx.DevBuf(4 * n), fdx.DevBuf(4 * n)
    fdx.check(fdx.lib.fdx_fold_layernorm_f32(None, None, fdx._dp(dw), fdx._dp(db), n, k, fdx._dp(wf), fdx._dp(ws), fdx._dp(bf)))
    fdx.check(fdx.lib.fdx_layernorm_dense_rows_f32(fdx._dp(dx), m, k, fdx.ctypes.c_float(1e-5), fdx._dp(wf), fdx._dp(ws), fdx._dp(bf), n,
                                                   None, None, fdx._dp(out)))
    d = (x64 - x64.mean(-1, keepdims=True)) / np.sqrt(x64.var(-1, keepdims=True) + 1e-5)
    # centring and scaling add a few roundings of each operand
    assert (np.abs(out.to_host((m, n)) - (d @ w64.T + b)) <= (steps + 24) * EPS * (np.abs(d) @ np.abs(w64).T + np.abs(b) + 1)).all()


@pytest.mark.parametrize("m", [3, 5, 6])
@pytest.mark.parametrize("k", [768, 3072])
def test_non_finite_rows_stay_their_own(fdx, m, k):
    x = np.ones((m, k), np.float32)
    x[m - 2, 5] = np.inf
    x[m - 1, k - 68] = np.nan
    w = np.random.default_rng(3).standard_normal((40, k)).astype(np.float32)
    dx, dw, out = fdx.DevBuf.from_host(x), fdx.DevBuf.from_host(w), fdx.DevBuf(4 * m * 40)
    fdx.check(fdx.lib.fdx_dense_rows_f32(fdx._dp(dx), m, k, fdx._dp(dw), None, 40, None, None, fdx._dp(out)))
    got = out.to_host((m, 40))
    assert np.isfinite(got[:m - 2]).all() and np.isinf(got[m - 2]).all() and np.isnan(got[m - 1]).all()
    assert (np.sign(got[m - 2]) == np.sign(w[:, 5])).all()


def test_more_columns_than_a_grid_holds(fdx):
    # 256 threads a column of a long row: 2^24 columns would be 2^32 threads, which the tile kernels' grid stays below
    form = fdx.lib.fdx_debug_dense_rows_form
    assert form(1, (1 << 24) - 1, 1028, 0) == 1 and form(1, 1 << 24, 1028, 0) == 0
