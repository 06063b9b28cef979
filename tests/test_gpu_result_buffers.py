"""Results written straight into the caller's device buffers: aligned and odd ones, buffers that meet the input or each other, results that
are views of inputs or that two outputs share, against the same model through host arrays."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Ptr:
    def __init__(self, buf, floats=0):
        self.buf, self.ptr = buf, ctypes.c_void_p(buf.ptr.value + 4 * floats)


def model(fdx, modelgen):
    b = modelgen.Builder("outs", 4)
    x = b.input((6, 6, 8), "in")
    y = b.conv2d(x, 8, 3, "a", padding="same", activation="relu", bias_std=0.1)   # read on by the rest and a result itself
    z = b.batchnorm(b.depthwise_conv2d(y, 3, "d", padding="same"), "bn", random_stats=True)
    f = b._add("Flatten", "f", {}, [z], (288,))                                   # a view
    return fdx.Model(modelgen.dumps(b.finish([y, f, b.dense(f, 5, "fc", activation="softmax")])), verify=False)


def run(fdx, m, x, outs):
    m.predict_dev(3, [x], [(6, 6, 8)], outs)
    fdx.sync()


@pytest.mark.parametrize("odd", [0, 1, 4])
def test_separate_buffers(fdx, modelgen, odd):
    m = model(fdx, modelgen)
    sizes = (288, 288, 5)
    for seed in (0, 1):   # the plan's own buffers are not confused by the first call's
        x = np.random.default_rng(seed).standard_normal((3, 6, 6, 8)).astype(np.float32)
        want = m.predict([x])
        d = fdx.DevBuf.from_host(x)
        bufs = [fdx.DevBuf.from_host(np.full(3 * n + 16, 9, np.float32)) for n in sizes]
        run(fdx, m, Ptr(d), [Ptr(t, odd) for t in bufs])
        for t, n, w in zip(bufs, sizes, want):
            h = t.to_host((3 * n + 16,))
            assert np.array_equal(h[odd:odd + 3 * n], w.reshape(-1))
            assert (h[:odd] == 9).all() and (h[odd + 3 * n:] == 9).all()
        assert np.array_equal(d.to_host(x.shape), x)
        again = m.predict([x])
        assert all(np.array_equal(a, b) for a, b in zip(want, again))


def test_result_over_the_input(fdx, modelgen):
    # "small": one launch, more samples than it has workgroups, which would write rows that others have still to read
    for shift in (0, 4, 400):
        for net in ("layers", "small"):
            b = modelgen.Builder("io", 6)
            x = b.input((6, 6, 8), "in")
            y = b.conv2d(x, 8, 3, "a", padding="same", activation="relu", bias_std=0.1)
            y = b.conv2d(y, 8, 3, "b", padding="same") if net == "small" else b.layernorm(y, "ln")
            m = fdx.Model(modelgen.dumps(b.finish([y])), verify=False)
            a = np.random.default_rng(2).standard_normal((300, 6, 6, 8)).astype(np.float32)
            fdx.lib.fdx_debug_force_sample_net(1)
            try:
                want = m.predict([a])[0]
                t = fdx.DevBuf.from_host(np.concatenate([a.reshape(-1), np.zeros(400, np.float32)]))
                m.predict_dev(300, [Ptr(t)], [(6, 6, 8)], [Ptr(t, shift)])
                fdx.sync()
                assert fdx.lib.fdx_debug_sample_net(m._h) == (net == "small")
            finally:
                fdx.lib.fdx_debug_force_sample_net(-1)
            assert np.array_equal(t.to_host((300 * 288 + 400,))[shift:shift + 300 * 288], want.reshape(-1)), (net, shift)


@pytest.mark.parametrize("shift", [4, 288, 860])
def test_results_that_meet_each_other(fdx, modelgen, shift):
    # the second one starts inside the first and ends beyond it: written one after the other, each whole
    m = model(fdx, modelgen)
    x = np.random.default_rng(7).standard_normal((3, 6, 6, 8)).astype(np.float32)
    y, f, c = [w.reshape(-1) for w in m.predict([x])]
    d, t, u = fdx.DevBuf.from_host(x), fdx.DevBuf.from_host(np.full(2 * 864, 9, np.float32)), fdx.DevBuf(4 * 16)
    run(fdx, m, Ptr(d), [Ptr(t), Ptr(t, shift), Ptr(u)])
    h = t.to_host((2 * 864,))
    assert np.array_equal(h[:shift], y[:shift]) and np.array_equal(h[shift:shift + 864], f) and (h[shift + 864:] == 9).all()
    assert np.array_equal(u.to_host((16,))[:15], c)


def test_two_outputs_of_one_layer_and_of_the_input(fdx, modelgen):
    b = modelgen.Builder("twice", 5)
    x = b.input((4, 4, 4), "in")
    y = b.conv2d(x, 4, 1, "a", activation="relu")
    m = fdx.Model(modelgen.dumps(b.finish([y, y, b._add("Flatten", "f", {}, [y], (64,)), b._add("Flatten", "g", {}, [x], (64,))])), verify=False)
    a = np.random.default_rng(3).standard_normal((2, 4, 4, 4)).astype(np.float32)
    want = m.predict([a])
    d, outs = fdx.DevBuf.from_host(a), [fdx.DevBuf(4 * 128) for _ in range(4)]
    m.predict_dev(2, [Ptr(d)], [(4, 4, 4)], [Ptr(t) for t in outs])
    fdx.sync()
    for t, w in zip(outs, want):
        assert np.array_equal(t.to_host((128,)), w.reshape(-1))
