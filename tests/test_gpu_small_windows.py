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
    import torch
    n, s, c = 3, 4096, 16  # 1 GiB an image
    x = torch.randn((n, s, s, c), device="cuda")
    w, b = torch.randn((3, 3, c), device="cuda"), torch.randn((c,), device="cuda")
    out, one = torch.full((n, s // 2, s // 2, c), 7.0, device="cuda"), torch.empty((1, s // 2, s // 2, c), device="cuda")
    torch.cuda.synchronize()
    p = lambda t, i=0: ctypes.c_void_p(t[i].data_ptr())

    def run(src, count, dst):
        fdx.check(fdx.lib.fdx_dwconv2d_nhwc_f32(src, count, s, s, c, ctypes.c_void_p(w.data_ptr()), ctypes.c_void_p(b.data_ptr()), 3, 3, 2, 2, 1, 1, 0, 0,
                                                s // 2, s // 2, None, dst))
        fdx.sync()

    run(p(x), n, p(out))
    for i in range(n):
        run(p(x, i), 1, p(one))
        assert torch.equal(one[0], out[i]), i
