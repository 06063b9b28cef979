"""Pooling over windows of 2 x 2 and 3 x 3 cells with all cells requested at once, at the edges of maps, against the oracle; depthwise
convolutions of tensors beyond 2 GiB, a launch to as many images as its offsets reach."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [2, 3])
@pytest.mark.parametrize("n,h,w,c,s", [(1, 1, 1, 4, 1), (2, 2, 3, 8, 1), (3, 7, 5, 12, 2), (1, 9, 10, 64, 3), (5, 4, 1, 4, 2), (2, 33, 31, 20, 2)])
@pytest.mark.parametrize("mode", ["max", "avg"])
def test_small_windows(fdx, oracle, n, h, w, c, s, k, mode):
    print("pool window", n, h, w, c, s, k, mode, flush=True)
    x = np.random.default_rng(7).standard_normal((n, h, w, c)).astype(np.float32) - 1
    for padding in ("same", "valid"):
        if padding == "valid" and (h < k or w < k):
            continue
        want = np.stack([oracle.pool2d(x[i], (k, k), (s, s), padding, mode) for i in range(n)])
        got = fdx.pool2d(x, (k, k), (s, s), padding, mode)
        assert got.shape == want.shape and np.abs(got - want).max() <= 1e-6  # up to nine values near 1 added in the same order
    framed = np.zeros((n, h + 3, w + 3, c), np.float32)  # one row above, two below, two columns left, one right
    framed[:, 1:1 + h, 2:2 + w] = x
    want = np.stack([oracle.pool2d(framed[i], (k, k), (s, s), "valid", mode) for i in range(n)])
    got = fdx.pool2d(x, (k, k), (s, s), "valid", mode, zero_frame=(1, 2, 2, 1))
    assert got.shape == want.shape and np.abs(got - want).max() <= 1e-6


def test_windows_of_infinities(fdx, oracle):
    x = np.full((1, 4, 4, 4), -np.inf, np.float32)
    x[0, 0, 0, 1] = np.inf
    x[0, 3, 3, 2] = 5
    for padding in ("same", "valid"):
        want = oracle.pool2d(x[0], (3, 3), (1, 1), padding, "max")
        assert np.array_equal(fdx.pool2d(x, (3, 3), (1, 1), padding, "max")[0], want)


def test_depthwise_beyond_two_gib(fdx):
    n, s, c = 3, 4096, 16  # 1 GiB an image
    r = np.random.default_rng(9)
    some = r.standard_normal(1 << 20).astype(np.float32)
    x = fdx.DevBuf(4 * n * s * s * c)
    for i in range(n):
        image = np.tile(np.roll(some, 77 * i), s * s * c >> 20)
        fdx.check(fdx.lib.fdx_h2d(ctypes.c_void_p(x.ptr.value + 4 * i * s * s * c), image.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(image.nbytes)))
    w, b = fdx.DevBuf.from_host(r.standard_normal((3, 3, c)).astype(np.float32)), fdx.DevBuf.from_host(r.standard_normal(c).astype(np.float32))
    size = 4 * s * s * c // 4
    out, one = fdx.DevBuf(n * size), fdx.DevBuf(size)

    def run(image, count, dst):
        fdx.check(fdx.lib.fdx_dwconv2d_nhwc_f32(ctypes.c_void_p(x.ptr.value + 4 * image * s * s * c), count, s, s, c, fdx._dp(w), fdx._dp(b), 3, 3, 2, 2, 1, 1, 0, 0,
                                                s // 2, s // 2, None, fdx._dp(dst)))

    run(0, n, out)
    got = out.to_host((n, size // 4))
    for i in range(n):
        run(i, 1, one)
        assert np.array_equal(one.to_host((size // 4,)), got[i]), i
