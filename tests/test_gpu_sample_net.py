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


@pytest.mark.parametrize("cin,cout,k,h", [(3, 16, 3, 16), (16, 16, 3, 12), (32, 32, 3, 8), (64, 56, 3, 5), (16, 16, 7, 8), (64, 32, 1, 8), (3, 8, 11, 16), (7, 33, 3, 8)])
def test_sums_as_close_to_64_bits_as_the_launches(fdx, modelgen, cin, cout, k, h):
    """A convolution's sums: sixteen products in a chain, such chunks by fours (one by one where channels are no multiple of four), then
    those.  A rounding is off by 2^-24 / sqrt(3) of the value at most in the root mean square; over a chain of n additions, whose sums grow
    like a square root, n / 2 of the last value's squared add up.  So 2^-24 / sqrt(3) sqrt(16 / 2 + 4 / 2 + chunks / 8 + 1), the one the bias;
    and no further off than a launch per layer."""
    b = modelgen.Builder("sums", 3)
    spec = b.finish([b.conv2d(b.input((h, h, cin), "in"), cout, k, "a", padding="same", bias_std=0.1)])
    p = spec["trainable_params"]["a"]
    w = np.asarray(p["weights"], np.float64).reshape(cout, k, k, cin)
    js = modelgen.dumps(spec)
    r = np.random.default_rng(21)
    for x in (r.standard_normal((64, h, h, cin)).astype(np.float32), r.uniform(0, 1, (64, h, h, cin)).astype(np.float32)):
        framed = np.pad(x.astype(np.float64), ((0, 0), (k // 2, k // 2), (k // 2, k // 2), (0, 0)))
        want = sum(framed[:, y:y + h, z:z + h] @ w[:, y, z].T for y in range(k) for z in range(k)) + p["bias"]
        err = {}
        for mode in (0, 1):
            fdx.lib.fdx_debug_force_sample_net(mode)
            try:
                model = fdx.Model(js, verify=False)
                got = model.predict([x])[0]
                assert fdx.lib.fdx_debug_sample_net(model._h) == mode
            finally:
                fdx.lib.fdx_debug_force_sample_net(-1)
            err[mode] = np.linalg.norm(got - want) / np.linalg.norm(want)
        chunks = -(-k * k * cin // 16)
        bound = 2.0 ** -24 / 3 ** 0.5 * np.sqrt(8 + (2 + chunks / 8 if cin % 4 == 0 else chunks / 2) + 1)
        print("sums", cin, cout, k, err, bound, flush=True)
        assert err[1] <= bound and err[1] <= err[0]


def test_refused_memory_leaves_the_launches(fdx, modelgen):
    js = modelgen.dumps(modelgen.small_cnn())
    x = np.random.default_rng(8).uniform(-1, 1, (3, 32, 32, 3)).astype(np.float32)
    want = fdx.Model(js, verify=False).predict([x])[0]
    fdx.lib.fdx_debug_fail_sample_memory(1)
    try:
        model = fdx.Model(js, verify=False)
        got = model.predict([x])[0]
        assert fdx.lib.fdx_debug_sample_net(model._h) == 0
        fdx.sync()
    finally:
        fdx.lib.fdx_debug_fail_sample_memory(0)
    assert rel(got, want) <= TOL


def test_a_program_goes_to_the_device_once_and_only_where_it_runs(fdx, modelgen):
    # two Dense layers of 128: the rule leaves batches beyond a few hundred to the launches
    b = modelgen.Builder("dense", 3)
    x = b.input((128,), "in")
    for i in range(2):
        x = b.dense(x, 128, "d%d" % i, activation="relu")
    model = fdx.Model(modelgen.dumps(b.finish([x])), verify=False)
    a = np.random.default_rng(4).standard_normal((2100, 128)).astype(np.float32)
    loads = fdx.lib.fdx_debug_sample_loads
    before = loads()
    for n in (2100, 2000, 1900, 1800, 1700, 1600):   # more batches than a model keeps plans
        model.predict([a[:n]])
        assert fdx.lib.fdx_debug_sample_net(model._h) == 0 and loads() == before, n
    want = model.predict([a[:1500]])[0]
    for n in (1, 2, 3, 4, 5, 6, 1):
        got = model.predict([a[:n]])[0]
        assert fdx.lib.fdx_debug_sample_net(model._h) == 1 and loads() == before + 1, n
        assert rel(got, want[:n]) <= TOL


def test_the_hook_tells_how_the_last_call_ran(fdx, modelgen):
    # a plan made for one launch, and a configuration of the layers' kernels forced behind it
    model = fdx.Model(modelgen.dumps(modelgen.small_cnn()), verify=False)
    x = np.random.default_rng(9).uniform(-1, 1, (5, 32, 32, 3)).astype(np.float32)
    want = model.predict([x])[0]
    assert fdx.lib.fdx_debug_sample_net(model._h) == 1
    fdx.check(fdx.lib.fdx_debug_force_tile(0))
    try:
        got = model.predict([x])[0]
        assert fdx.lib.fdx_debug_sample_net(model._h) == 0
    finally:
        fdx.check(fdx.lib.fdx_debug_force_tile(-1))
    assert rel(got, want) <= TOL
    model.predict([x])
    assert fdx.lib.fdx_debug_sample_net(model._h) == 1


@pytest.mark.parametrize("net,shape,batch", [("small_cnn", (32, 32, 3), 401), ("small_cnn", (32, 32, 3), 1030), ("odd_input", (61, 47, 5), 77), ("odd_input", (61, 47, 5), 1111)])
def test_host_arrays_in_pieces(fdx, modelgen, net, shape, batch):
    """From 4 MB on host arrays arrive in pieces, and each piece runs behind its copy: the bits of the whole batch in device memory.  Pieces below
    and above a round of workgroups, a last piece of its own size, samples that are no multiple of 16 bytes, more than 16 MB a quarter."""
    if net == "small_cnn":
        js = modelgen.dumps(modelgen.small_cnn())
    else:
        b = modelgen.Builder(net, 11)
        js = modelgen.dumps(b.finish([NETS[net](b)]))
    x = np.random.default_rng(batch).uniform(-1, 1, (batch,) + shape).astype(np.float32)
    assert x.nbytes >= 4 << 20
    fdx.lib.fdx_debug_force_sample_net(1)
    try:
        model = fdx.Model(js, verify=False)
        n = int(np.prod(model.output_shapes[0]))
        got = [model.predict([x])[0], model.predict_samples([[a] for a in x])[0]]
        assert fdx.lib.fdx_debug_sample_net(model._h) == 1
        d, out = fdx.DevBuf.from_host(x), fdx.DevBuf(4 * batch * n)
        model.predict_dev(batch, [d], [shape], [out])
        fdx.sync()
        want = out.to_host((batch, n))
    finally:
        fdx.lib.fdx_debug_force_sample_net(-1)
    for g in got:
        assert np.array_equal(np.asarray(g).reshape(batch, n), want)


def test_the_rule_follows_the_layers_own_times(fdx, modelgen):
    """Two convolutions of 5x5 / 2 and 3x3 to 24 and 64 channels on 12 x 12: as one launch twice as fast up to a few hundred samples, twice as slow
    for 8192 (267 us against 126).  Three convolutions with six channels in the middle on 8 x 8: 13 against 44 us for one sample."""
    def wide(b):
        return b.conv2d(b.conv2d(b.input((12, 12, 8), "in"), 24, 5, "a", strides=2, padding="same", activation="relu"), 64, 3, "b", padding="same")

    def thin(b):
        x = b.conv2d(b.input((8, 8, 4), "in"), 48, 3, "a", padding="same", activation="relu")
        x = b.pool(b.conv2d(x, 6, 3, "b", padding="same", activation="relu"), "p", 2, 2)
        return b.conv2d(x, 48, 5, "c", padding="same")

    for f, shape, forms in ((wide, (12, 12, 8), {1: 1, 64: 1, 8192: 0}), (thin, (8, 8, 4), {1: 1, 256: 1})):
        b = modelgen.Builder(f.__name__, 3)
        model = fdx.Model(modelgen.dumps(b.finish([f(b)])), verify=False)
        for n, form in forms.items():
            model.predict([np.zeros((n,) + shape, np.float32)])
            assert fdx.lib.fdx_debug_sample_net(model._h) == form, (f.__name__, n)
