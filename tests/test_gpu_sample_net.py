"""Small models as one launch (a workgroup takes a sample through every layer) against the oracle and against a launch per layer.
Sums of K products in another order differ by at most K rounding errors of the sum of magnitudes; a few layers of unit-variance
operands stay far below 1e-5 of the largest output, which is the bound here (1e-4 is the contract)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-5


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    assert a.shape == b.shape, (a.shape, b.shape)
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-30)


def odd_convs(b):
    # channels that are no multiple of four, ragged maps, strides, dilation, a wide frame; the result is a map
    x = b.input((13, 9, 3), "in")
    x = b.conv2d(x, 5, (5, 3), "a", padding="same", activation="relu", bias_std=0.2)
    x = b.conv2d(x, 7, 3, "b", padding="same", dilation=2, activation="gelu", bias_std=0.2)
    x = b.conv2d(x, 18, 3, "c", strides=2, padding="valid")
    return b.conv2d(x, 33, 1, "d", activation="relu", bias_std=0.1)


def residual(b):
    x = b.input((8, 8, 8), "in")
    x = b.conv2d(x, 16, 3, "a", padding="same", activation="relu")
    y = b.conv2d(x, 16, 3, "b", padding="same", activation="relu")
    y = b.conv2d(y, 16, 3, "c", padding="same")
    x = b.relu(b.add([x, y], "add"), "r")
    x = b.pool(x, "p", 3, 2, padding="same", kind="avg")
    x = b.pool(x, "q", 2, 1, padding="same")
    x = b.gap(x, "g", kind="max")
    return b.dense(x, 3, "fc", activation="softmax", bias_std=0.3)


def flattened(b):
    # Flatten behind a pooling layer: the tensor is read as one run
    x = b.input((12, 12, 1), "in")
    x = b.conv2d(x, 6, 5, "a", padding="same", activation="tanh")
    x = b.pool(x, "p", 2, 2)
    x = b.conv2d(x, 16, 3, "b", activation="relu", bias_std=0.1)
    x = b.pool(x, "q", 2, 2)
    x = b._add("Flatten", "f", {}, [x], (64,))
    x = b.dense(x, 40, "d1", activation="relu", bias_std=0.1)
    return b.dense(x, 17, "d2", activation="sigmoid")


def sequence(b):
    x = b.input((21, 6), "in")
    x = b.dense(x, 40, "a", activation="gelu", bias_std=0.2)
    return b.dense(x, 70, "b", activation="softmax")


def wide_pool(b):
    x = b.input((3, 5, 2), "in")
    x = b.conv2d(x, 1100, 1, "a", activation="relu", bias_std=0.3)
    return b.gap(x, "g")


def vectors(b):
    # matrices times one pixel: odd K, more rows than a workgroup takes at once, a K of several rounds; pooled channels that are no
    # multiple of four; 2 x 2 windows that leave a row and a column over
    x = b.input((9, 7, 8), "in")
    x = b.pool(x, "p", 2, 2)
    x = b.conv2d(x, 13, 3, "a", padding="same", activation="relu", bias_std=0.2)
    x = b.gap(x, "g")
    x = b.dense(x, 150, "b", activation="relu", bias_std=0.3)
    x = b.dense(x, 68, "c", activation="gelu", bias_std=0.3)
    return b.dense(x, 5, "d", bias_std=0.1)


def full_input(b):
    # the largest input
    x = b.pool(b.input((64, 64, 4), "in"), "p", 4, 4)
    return b.gap(b.conv2d(x, 20, 3, "a", activation="relu", bias_std=0.2), "g")


def odd_input(b):
    # a volume that is no multiple of four
    x = b.pool(b.input((61, 47, 5), "in"), "p", 3, 3, kind="avg")
    return b.gap(b.conv2d(x, 6, 3, "a", activation="relu", bias_std=0.2), "g", kind="max")


NETS = {f.__name__: f for f in (odd_convs, residual, flattened, sequence, wide_pool, vectors, full_input, odd_input)}


@pytest.mark.parametrize("batch", [1, 3, 300])  # one sample, fewer than CUs, more than CUs (a workgroup's second sample)
@pytest.mark.parametrize("net", list(NETS) + ["small_cnn"])
def test_small_model_as_one_launch(fdx, oracle, modelgen, net, batch):
    print("sample net", net, batch, flush=True)
    if net == "small_cnn":
        spec = modelgen.small_cnn()
    else:
        b = modelgen.Builder(net, 11)
        spec = b.finish([NETS[net](b)])
    js = modelgen.dumps(spec)
    ref = oracle.OracleModel(js)
    shape = tuple(d for d in spec["input_shapes"][0] if d is not None) if "input_shapes" in spec else None
    r = np.random.default_rng(batch)
    x = r.uniform(-1, 1, (batch,) + shape).astype(np.float32)
    got = {}
    for mode in (0, 1):
        fdx.lib.fdx_debug_force_sample_net(mode)
        try:
            model = fdx.Model(js, verify=False)
            got[mode] = model.predict([x])[0]
            assert fdx.lib.fdx_debug_sample_net(model._h) == mode
            if mode == 1:
                again = model.predict([x[:1]])[0]
                assert np.array_equal(again, got[1][:1])   # a sample's result does not depend on its neighbours
        finally:
            fdx.lib.fdx_debug_force_sample_net(-1)
    assert rel(got[1], got[0]) <= TOL
    for i in {0, batch // 2, batch - 1}:
        assert rel(got[1][i], ref.predict([x[i]])[0]) <= TOL, i


def test_non_finite_samples_stay_their_own(fdx, modelgen):
    # infinities and NaN pass through as in the layers' own launches, and touch no other sample; padding and the zeros behind K
    # meet them without turning them into NaN
    js = modelgen.dumps(modelgen.small_cnn())
    x = np.random.default_rng(5).uniform(-1, 1, (4, 32, 32, 3)).astype(np.float32)
    x[1, 3, 3, 0] = np.inf
    x[2, 31, 31, 2] = np.nan
    out = {}
    for mode in (0, 1):
        fdx.lib.fdx_debug_force_sample_net(mode)
        try:
            out[mode] = fdx.Model(js, verify=False).predict([x])[0]
        finally:
            fdx.lib.fdx_debug_force_sample_net(-1)
    assert np.isfinite(out[1][[0, 3]]).all()
    assert np.array_equal(np.isnan(out[0]), np.isnan(out[1]))
    assert rel(out[1][[0, 3]], out[0][[0, 3]]) <= TOL


def test_models_without_a_program_keep_their_launches(fdx, modelgen):
    # weights beyond a CU's LDS, an operation without a step, an input beyond the registers
    def big(b):
        return b.dense(b.input((300,), "in"), 300, "a")

    def norm(b):
        return b.layernorm(b.input((5, 8), "in"), "a")

    def wide(b):
        return b.gap(b.conv2d(b.input((80, 80, 3), "in"), 4, 3, "a"), "g")

    fdx.lib.fdx_debug_force_sample_net(1)
    try:
        for f, shape in ((big, (300,)), (norm, (5, 8)), (wide, (80, 80, 3))):
            b = modelgen.Builder(f.__name__, 3)
            model = fdx.Model(modelgen.dumps(b.finish([f(b)])), verify=False)
            model.predict([np.zeros((2,) + shape, np.float32)])
            assert fdx.lib.fdx_debug_sample_net(model._h) == 0, f.__name__
    finally:
        fdx.lib.fdx_debug_force_sample_net(-1)
