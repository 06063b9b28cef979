"""The kernel for problems with few output tiles (configurations 40-44: the waves of a workgroup cut one tile's K range
between them), against fp64 products.  fp32 products summed in another order differ by at most K rounding errors of the sum
of magnitudes, K 2^-24; operands of unit variance keep the typical error far below it, so 2e-6 relative to the largest
output leaves a factor of four over what the largest K here shows."""
import zlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 2e-6


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    assert a.shape == b.shape, (a.shape, b.shape)
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-30)


@pytest.mark.parametrize("tile", [-1, 40, 41, 42, 43, 44])
@pytest.mark.parametrize("m,n,k", [(1, 16, 16), (1, 1000, 2048), (15, 20, 48), (16, 64, 32), (17, 36, 112), (33, 96, 160), (49, 512, 4608),
                                   (65, 68, 512), (231, 132, 272), (700, 24, 144)])
def test_gemm_few_tiles(fdx, m, n, k, tile):
    print("gemm few tiles", m, n, k, tile, flush=True)
    r = np.random.default_rng(zlib.crc32(repr((m, n, k)).encode()))
    a, w = r.standard_normal((m, k)).astype(np.float32), (r.standard_normal((n, k)) / np.sqrt(k)).astype(np.float32)
    b, res = r.standard_normal(n).astype(np.float32), r.standard_normal((m, n)).astype(np.float32)
    want = a.astype(np.float64) @ w.astype(np.float64).T
    fdx.lib.fdx_debug_force_tile(tile)
    try:
        plain = fdx.gemm(a, w)
        full = fdx.gemm(a, w, b, alpha=0.5, residual=res, act=fdx.relu_act(1.5))
        again = fdx.gemm(a, w, b, alpha=0.5, residual=res, act=fdx.relu_act(1.5))
    finally:
        fdx.lib.fdx_debug_force_tile(-1)
    assert rel(plain, want) <= TOL
    assert rel(full, np.clip(0.5 * want + b + res, 0, 1.5)) <= TOL
    assert np.array_equal(full, again)  # the waves' partial tiles are added in wave order


@pytest.mark.parametrize("tile", [-1, 40, 41, 42, 43, 44])
@pytest.mark.parametrize("case", [
    # n, h, w, cin, cout, kh, kw, strides, dilation, padding
    (1, 7, 7, 512, 64, 3, 3, (1, 1), (1, 1), "same"),
    (2, 9, 7, 48, 20, 3, 3, (1, 1), (1, 1), "same"),     # 16-k units: channels no multiple of 32, ragged rows and columns
    (1, 14, 14, 64, 32, 1, 1, (2, 2), (1, 1), "valid"),
    (1, 12, 13, 32, 12, 2, 3, (1, 1), (2, 3), "same"),   # dilation
    (3, 15, 15, 16, 36, 3, 3, (2, 1), (1, 1), "valid"),
    (1, 3, 2, 16, 16, 5, 5, (1, 1), (1, 1), "same"),     # most taps outside the image
])
def test_conv2d_few_tiles(fdx, oracle, case, tile):
    n, h, w, cin, cout, kh, kw, strides, dilation, padding = case
    print("conv2d few tiles", case, tile, flush=True)
    r = np.random.default_rng(zlib.crc32(repr(case).encode()))
    x = r.standard_normal((n, h, w, cin)).astype(np.float32)
    wj = (r.standard_normal((cout, kh, kw, cin)) / np.sqrt(kh * kw * cin)).astype(np.float32)
    b = r.standard_normal(cout).astype(np.float32)
    wo = oracle.conv2d_prepare(wj, cout, kh, kw, cin)
    conv = np.stack([oracle.conv2d(x[i], wo, b, cout, kh, kw, strides, dilation, padding) for i in range(n)])
    res = r.standard_normal(conv.shape).astype(np.float32)
    fdx.lib.fdx_debug_force_tile(tile)
    try:
        got = fdx.conv2d(x, wj, b, strides, dilation, padding, residual=res, act=fdx.relu_act())
    finally:
        fdx.lib.fdx_debug_force_tile(-1)
    assert rel(got, oracle.relu(oracle.add(res, conv))) <= 2 * TOL  # the oracle sums in fp32 as well


@pytest.mark.parametrize("tile", [-1, 40, 42, 44])
def test_residual_block_with_shortcut_convolution_few_tiles(fdx, oracle, modelgen, tile):
    """Two convolutions summed as one GEMM over both inputs' channels (strided shortcut), at a batch of one."""
    b = modelgen.Builder("dual", 5)
    x = b.input((14, 14, 64), "x")
    y = b.conv2d(x, 32, 1, "c1", strides=2, activation="relu", bias_std=0.1)
    y = b.conv2d(y, 48, 1, "c2", bias_std=0.1)
    s = b.conv2d(x, 48, 1, "c0", strides=2, bias_std=0.1)
    js = modelgen.dumps(b.finish([b.add([s, y], "sum")]))
    xs = np.random.default_rng(6).standard_normal((1, 14, 14, 64)).astype(np.float32)
    want = oracle.OracleModel(js).predict([xs[0]])[0][None]
    fdx.lib.fdx_debug_force_tile(tile)
    try:
        got = fdx.Model(js, verify=False).predict([xs])[0]
    finally:
        fdx.lib.fdx_debug_force_tile(-1)
    assert rel(got, want) <= 2 * TOL


@pytest.mark.parametrize("tile", [40, 41, 42, 43, 44])
@pytest.mark.parametrize("mid,cin,n,size", [(16, 48, 1, 9), (48, 16, 3, 5), (48, 80, 1, 14), (32, 64, 2, 7), (160, 32, 1, 3)])
def test_both_units_of_the_two_source_form(fdx, oracle, modelgen, tile, mid, cin, n, size):
    """The sum of two pointwise convolutions as one GEMM: channel counts that are multiples of 16 only (the 16-float unit) and
    of 32 (the 32-float one) in either source, waves whose share of K lies in one source, in both, or is empty."""
    print("two sources", tile, mid, cin, n, size, flush=True)
    b = modelgen.Builder("dual", 15)
    x = b.input((size, size, cin), "x")
    y = b.conv2d(x, mid, 1, "c1", strides=2, activation="relu", bias_std=0.1)
    y = b.conv2d(y, 52, 1, "c2", bias_std=0.1)
    s = b.conv2d(x, 52, 1, "c0", strides=2, bias_std=0.1)
    js = modelgen.dumps(b.finish([b.add([s, y], "sum")]))
    xs = np.random.default_rng(16).standard_normal((n, size, size, cin)).astype(np.float32)
    ref = oracle.OracleModel(js)
    want = np.stack([ref.predict([xs[i]])[0] for i in range(n)])
    model = fdx.Model(js, verify=False)
    fdx.lib.fdx_debug_force_tile(tile)
    try:
        got = model.predict([xs])[0]
        again = model.predict([xs])[0]
    finally:
        fdx.lib.fdx_debug_force_tile(-1)
    assert rel(got, want) <= 2 * TOL
    assert np.array_equal(got, again)


def test_more_tiles_than_a_launch_can_hold(fdx):
    """131072 x 16384 outputs (8.6 GB): a workgroup of 512 threads for each 16 x 16 of them would be 2^32 threads.  Neither
    the timing runs nor a forced form takes that form."""
    m, n, k = 131072, 16384, 16
    c = fdx.ctypes
    print("gemm", m, n, k, flush=True)
    r = np.random.default_rng(12)
    a, w = r.standard_normal((m, k)).astype(np.float32), r.standard_normal((n, k)).astype(np.float32)
    da, dw, out = fdx.DevBuf.from_host(a), fdx.DevBuf.from_host(w), fdx.DevBuf(4 * m * n)
    rows = [0, 1, m // 2, m - 1]
    got = np.empty((len(rows), n), np.float32)
    for timing, tile in ((False, -1), (False, 40), (True, -1), (True, -1)):
        fdx.tuner_timing(timing)
        fdx.lib.fdx_debug_force_tile(tile)
        try:
            fdx.check(fdx.lib.fdx_gemm_bias_act_f32(fdx._dp(da), c.c_int64(k), fdx._dp(dw), c.c_int64(k), m, n, k, c.c_float(1), None, 0, None,
                                                    None, fdx._dp(out), c.c_int64(n), None))
            fdx.sync()
        finally:
            fdx.lib.fdx_debug_force_tile(-1)
            fdx.tuner_timing(False)
        for i, row in enumerate(rows):
            fdx.check(fdx.lib.fdx_d2h(got[i].ctypes.data_as(c.c_void_p), c.c_void_p(out.ptr.value + 4 * n * row), c.c_size_t(4 * n)))
        assert rel(got, a[rows].astype(np.float64) @ w.astype(np.float64).T) <= TOL
