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
                                     (130, 3, 3, 128), (2, 9, 5, 67),
                                     # both sides of the lines to the form for few positions, every number of its last loads
                                     (3, 8, 8, 64), (3, 5, 13, 64), (3, 4, 8, 63), (3, 3, 11, 63), (700, 2, 2, 130), (2, 1, 2, 200), (2, 1, 3, 64),
                                     (2, 1, 5, 12), (2, 3, 3, 65), (2, 13, 1, 96), (2, 1, 17, 64), (2, 3, 7, 64)])
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


@pytest.mark.parametrize("rows,depth", [(999, 257), (1000, 257), (1001, 512), (1999, 513), (2000, 513), (2003, 1024), (5000, 300), (2000, 1025)])
def test_softmax_many_rows(fdx, oracle, rows, depth):
    """Rows of 257 to 1024 entries on both sides of the lines between a workgroup and a wave per row."""
    print("softmax many rows", rows, depth, flush=True)
    x = np.random.default_rng(6).normal(0, 3, (rows, depth)).astype(np.float32)
    x[-1, -1] = 60.0
    # at most depth roundings of 2^-24 in the sum, a few units in the last place of expf and logf on each side
    assert rel(fdx.softmax(x), oracle.softmax(x)) <= 1e-5
    t = min(rows, 7)
    got = fdx.softmax(x[: rows // t * t], causal_period=t, causal_offset=depth - t)
    for row in (0, 1, rows // t * t - 1):
        visible = row % t + 1 + depth - t
        assert rel(got[row, :visible], oracle.softmax(x[row, :visible])) <= 1e-5
        assert not got[row, visible:].any()


def test_softmax_of_more_rows_than_a_launch_has_workgroups_of_256(fdx, oracle):
    """2^24 rows and more of 257 entries (17 GB, in place): a workgroup of 256 threads for each would be 2^32 threads.  The
    rows looked at are written, the others hold whatever the memory held."""
    c = fdx.ctypes
    rows, depth = (1 << 24) + 3, 257
    print("softmax", rows, depth, flush=True)
    buf = fdx.DevBuf(4 * rows * depth)
    at = [0, 1, 4095, (1 << 23) + 1, (1 << 24) - 1, 1 << 24, rows - 1]
    x = np.random.default_rng(7).normal(0, 3, (len(at), depth)).astype(np.float32)
    got = np.empty_like(x)
    place = lambda i: c.c_void_p(buf.ptr.value + 4 * depth * at[i])
    for i in range(len(at)):
        fdx.check(fdx.lib.fdx_h2d(place(i), x[i].ctypes.data_as(c.c_void_p), c.c_size_t(4 * depth)))
    fdx.check(fdx.lib.fdx_softmax_f32(fdx._dp(buf), c.c_int64(rows), depth, 0, 0, fdx._dp(buf)))
    for i in range(len(at)):
        fdx.check(fdx.lib.fdx_d2h(got[i].ctypes.data_as(c.c_void_p), place(i), c.c_size_t(4 * depth)))
    assert rel(got, oracle.softmax(x)) <= 1e-5


@pytest.mark.parametrize("t,s", [(3, 60), (5, 200), (7, 700)])
def test_softmax_causal(fdx, oracle, t, s):
    print("softmax causal", t, s, flush=True)
    x = np.random.default_rng(5).normal(0, 2, (2 * t, s)).astype(np.float32)
    got = fdx.softmax(x, causal_period=t, causal_offset=s - t)
    for row in range(2 * t):
        visible = row % t + 1 + s - t
        assert rel(got[row, :visible], oracle.softmax(x[row, :visible])) <= 1e-5
        assert not got[row, visible:].any()
