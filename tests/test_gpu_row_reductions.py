"""Global pooling and softmax at the edges of their kernels' forms: channel counts with and without the 16-byte form, fewer
and more positions than slots, rows at the ends of the ranges that stay in registers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    assert a.shape == b.shape, (a.shape, b.shape)
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-30)


@pytest.mark.parametrize("n,h,w,c", [(1, 1, 1, 4), (2, 7, 7, 1), (1, 16, 16, 32), (3, 5, 13, 30), (1, 7, 7, 2048), (5, 33, 31, 68),
                                     (130, 3, 3, 128), (2, 9, 5, 67)])
@pytest.mark.parametrize("mode", ["avg", "max"])
def test_global_pool(fdx, oracle, n, h, w, c, mode):
    print("global pool", n, h, w, c, mode, flush=True)
    x = np.random.default_rng(3).normal(-2, 1, (n, h, w, c)).astype(np.float32)
    want = np.stack([oracle.global_pool(x[i], mode) for i in range(n)])
    got = fdx.global_pool(x, mode)
    if mode == "max":
        assert np.array_equal(got, want)
    else:
        # both sides take at most h * w roundings of 2^-24; the terms' magnitudes add up to at most 1.2 times the sums
        assert rel(got, want) <= 2.0 ** -24 * 1.2 * (2 * h * w + 2)


@pytest.mark.parametrize("rows", [1, 5, 300])
@pytest.mark.parametrize("depth", [1, 63, 64, 65, 256, 257, 1000, 1024, 1025])
def test_softmax(fdx, oracle, rows, depth):
    print("softmax", rows, depth, flush=True)
    x = np.random.default_rng(4).normal(0, 3, (rows, depth)).astype(np.float32)
    x[0, 0] = -np.inf if depth > 1 else 0.0
    x[-1, depth // 2] = 80.0
    assert rel(fdx.softmax(x), oracle.softmax(x)) <= 1e-5


@pytest.mark.parametrize("t,s", [(3, 60), (5, 200), (7, 700)])
def test_softmax_causal(fdx, oracle, t, s):
    print("softmax causal", t, s, flush=True)
    x = np.random.default_rng(5).normal(0, 2, (2 * t, s)).astype(np.float32)
    got = fdx.softmax(x, causal_period=t, causal_offset=s - t)
    for row in range(2 * t):
        visible = row % t + 1 + s - t
        assert rel(got[row, :visible], oracle.softmax(x[row, :visible])) <= 1e-5
        assert not got[row, visible:].any()
