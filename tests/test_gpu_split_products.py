"""The tiled GEMM / convolution kernel (configurations 13-18, cut along K in several ways): fp32 operands as exact sums of three
bf16 values on the bf16 matrix instructions.

Error bound: every 16 steps of K round the main sum once (at most 2^-24 of the running sum, itself at most the sum of the
magnitudes S); the products left out are at most 2^-24 S (the second part of a value is at most 2^-8 of it, the third 2^-17, so
a1 b2 and a2 b1 are 2^-25 of a b each; 2^-27.5 on average); bias, residual, the sum with the small products and those of partial
tiles round a few times more, seven are allowed for; twice all that: (K / 16 + 8) 2^-23 S for an element.  For the 2-norm, where roundings average out, twice what operands of
unit variance show against 64 bits (6e-9 sqrt(K))."""
import zlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TILES = [-1, 13, 14, 15, 16, 18, 215, 815, 315 + 10000, 20013, 20015]
HALO = [23, 24, 28, 223]


def forced(fdx, tile, f):
    fdx.lib.fdx_debug_force_tile(tile)
    try:
        return f()
    finally:
        fdx.lib.fdx_debug_force_tile(-1)


def check(got, a, w, extra=0.0):
    a, w = a.astype(np.float64), w.astype(np.float64)
    want, size, k = a @ w.T + extra, np.abs(a) @ np.abs(w).T + np.abs(extra), a.shape[1]
    err = np.abs(got - want)
    assert (err <= (k / 16 + 8) * 2.0 ** -23 * size).all(), (err / size).max()
    assert np.linalg.norm(err) <= (1.2e-8 * np.sqrt(k) + 1.2e-7) * np.linalg.norm(want)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("m,n,k", [(1, 36, 16), (63, 64, 48), (129, 132, 32), (255, 100, 272), (257, 260, 512), (640, 64, 2320)])
def test_gemm_edges(fdx, m, n, k, tile):
    print("split products", m, n, k, tile, flush=True)
    r = np.random.default_rng(zlib.crc32(repr((m, n, k)).encode()))
    a, w = r.standard_normal((m, k)).astype(np.float32), (r.standard_normal((n, k)) / np.sqrt(k)).astype(np.float32)
    b, res = r.standard_normal(n).astype(np.float32), r.standard_normal((m, n)).astype(np.float32)
    plain, full, again = forced(fdx, tile, lambda: (fdx.gemm(a, w), fdx.gemm(a, w, b, residual=res), fdx.gemm(a, w, b, residual=res)))
    check(plain, a, w)
    check(full, a, w, (b + res).astype(np.float64))
    assert np.array_equal(full, again)
    # the split does not depend on the operands' scale
    scaled = forced(fdx, tile, lambda: fdx.gemm(a * np.float32(2.0 ** 60), w * np.float32(2.0 ** -50)))
    assert np.array_equal(scaled, plain * np.float32(2.0 ** 10))


@pytest.mark.parametrize("tile", [13, 14, 15, 16, 18, 215, 20013])
@pytest.mark.parametrize("k", [16, 352])
def test_left_out_products_that_add_up(fdx, tile, k):
    """All operands close to 1 + 2^-8 - 2^-17, whose parts are the largest there are and have one sign: the products left out are
    2^-24.02 of every product and do not average out.  Undoubled bound of an element."""
    print("left out products", tile, k, flush=True)
    r = np.random.default_rng(12)
    m, n = 130, 68
    near = lambda *shape: (float.fromhex("0x1.00fe8p0") + r.integers(-2, 3, shape) * 2.0 ** -23).astype(np.float32)
    a, w = near(m, k), near(n, k)
    got = forced(fdx, tile, lambda: fdx.gemm(a, w))
    want = a.astype(np.float64) @ w.astype(np.float64).T
    assert (np.abs(got - want) <= (k / 16 + 8) * 2.0 ** -24 * want).all()


# exponents of A's and of W's values: one side, or both, around the smallest normal and among the subnormal numbers
@pytest.mark.parametrize("ea,ew", [(-122, 110), (110, -122), (-127, 115), (-140, 120), (120, -140), (-75, -65)])
@pytest.mark.parametrize("tile", [13, 14, 15, 16, 18, 215, 20013] + HALO)
def test_tiny_operands(fdx, tile, ea, ew):
    """Operands whose last bits lie below bf16's range keep all of them: the bound of ordinary operands.  (Results below 2^-126
    are rounded once to multiples of 2^-149, which the last term allows; the kernels on fp32 instructions, which the closed rule
    takes for a problem as small as this, round every partial sum there.)"""
    print("tiny operands", tile, ea, ew, flush=True)
    r = np.random.default_rng(11)
    m, n, k = 130, 68, 352
    a = np.ldexp(r.standard_normal((m, k)), ea).astype(np.float32)
    w = np.ldexp(r.standard_normal((n, k)) / np.sqrt(k), ew).astype(np.float32)
    if tile in HALO:   # a 1x3 filter over rows of 130 positions, only its middle tap not zero
        wc = np.zeros((n, 1, 3, k), np.float32)
        wc[:, 0, 1] = w
        got = forced(fdx, tile, lambda: fdx.conv2d(a.reshape(1, 1, m, k), wc, None, padding="same")).reshape(m, n)
    else:
        got = forced(fdx, tile, lambda: fdx.gemm(a, w))
    a, w = a.astype(np.float64), w.astype(np.float64)
    want, size = a @ w.T, np.abs(a) @ np.abs(w).T
    assert (np.abs(got - want) <= (k / 16 + 8) * 2.0 ** -23 * size + 2.0 ** -148).all(), (np.abs(got - want) / size).max()


def special(a, w):
    a[1, 3], a[2, -1], a[3, 0], a[4, 5] = np.inf, -np.inf, np.nan, 3.4e38   # 3.4e38 rounds up to an infinite bf16
    a[5, 2], a[5, -2] = np.inf, -np.inf
    w[0, 1], w[2, -3] = np.inf, np.nan
    w[3, :] = 0                                                            # 0 * Inf
    w[4, 5] = 0.25


def check_special(got, a, w):
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ w.astype(np.float64).T
        want = np.where(np.abs(want) > np.finfo(np.float32).max, np.sign(want) * np.inf, want)
    finite = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[~finite & ~np.isnan(want)], want[~finite & ~np.isnan(want)])
    assert np.allclose(got[finite], want[finite], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("tile", TILES + HALO)
def test_infinities_and_nan(fdx, tile):
    print("special operands", tile, flush=True)
    r = np.random.default_rng(5)
    m, n, k = 140, 68, 352
    a, w = r.standard_normal((m, k)).astype(np.float32), (r.standard_normal((n, k)) / 18).astype(np.float32)
    special(a, w)
    check_special(forced(fdx, tile, lambda: fdx.gemm(a, w)), a, w)
    # a 3x3 convolution over a map of ten positions a row: the same products with zero taps around
    x = a.reshape(1, m // 10, 10, k).copy()
    wc = np.zeros((n, 3, 3, k), np.float32)
    wc[:, 1, 1] = w
    got = forced(fdx, tile, lambda: fdx.conv2d(x, wc, None, padding="same")).reshape(m, n)
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ w.astype(np.float64).T
    far = np.ones(m, bool)
    far[:20] = False                      # zero taps of the neighbours meet infinities there: only positions past them compare
    far_w = np.isfinite(w).all(1)
    assert np.allclose(got[far][:, far_w], want[far][:, far_w], rtol=1e-4, atol=1e-4)
    assert np.isnan(got[:, 2]).all() and not np.isfinite(got[far][:, 0]).any()


def test_infinities_two_sources(fdx, modelgen):
    """The sum of two 1x1 convolutions as one GEMM: an infinite pixel of either map gives that pixel's infinities and nothing else."""
    b = modelgen.Builder("two_src", 7)
    x = b.input((9, 7, 32), "img")
    y = b.conv2d(x, 16, 1, "c1", strides=2, use_bias=False)
    z = b.conv2d(y, 64, 1, "c3", bias_std=0.2)
    sc = b.conv2d(x, 64, 1, "sc", strides=2, bias_std=0.1)
    spec = b.finish([b.add([sc, z], "sum")])
    xs = np.random.default_rng(3).standard_normal((4, 9, 7, 32)).astype(np.float32)
    bad = xs.copy()
    bad[2, 4, 2, 5] = np.inf
    print("two sources", flush=True)
    model = fdx.Model(modelgen.dumps(spec), verify=False)
    for tile in (-1, 13, 14, 15, 16, 18):
        want, got = forced(fdx, tile, lambda: (model.predict([xs])[0], model.predict([bad])[0]))
        hit = np.zeros(want.shape[:3], bool)
        hit[2, 2, 1] = True
        assert np.array_equal(got[~hit], want[~hit]) and not np.isfinite(got[hit]).any()


def test_infinities_rows_shorter_than_k(fdx, modelgen):
    """A 1x1 convolution over 24 channels reads rows of 32, the last 8 of the next pixel: an infinite pixel stays alone."""
    b = modelgen.Builder("short_rows", 8)
    x = b.input((9, 14, 24), "img")
    spec = b.finish([b.conv2d(x, 144, 1, "c", bias_std=0.2)])
    xs = np.random.default_rng(4).standard_normal((5, 9, 14, 24)).astype(np.float32)
    bad = xs.copy()
    bad[3, 4, 2, 5], bad[4, 8, 13, 23], bad[1, 2, 3, 0] = np.inf, np.nan, 3e38
    model = fdx.Model(modelgen.dumps(spec), verify=False)
    hit = np.zeros(xs.shape[:3], bool)
    hit[3, 4, 2] = hit[4, 8, 13] = hit[1, 2, 3] = True
    for tile in (13, 14, 15, 16, 18):
        print("short rows", tile, flush=True)
        want, got = forced(fdx, tile, lambda: (model.predict([xs])[0], model.predict([bad])[0]))
        # (the pixels in front of these meet them with zero taps and are summed again, in another order)
        assert np.allclose(got[~hit], want[~hit], rtol=1e-5, atol=1e-5) and not np.isfinite(got[3, 4, 2]).any() and np.isnan(got[4, 8, 13]).all()


def test_time_of_not_finite_operands(fdx):
    """Sums that are taken again cost a few times what finite ones do (1.4 times the GEMM, 2.5 the convolution, 2.3 attention;
    one lane per element took 150 to 350 times): eight times is allowed for a busy machine."""
    import ctypes
    r = np.random.default_rng(6)
    dev = lambda *shape: fdx.DevBuf.from_host(r.standard_normal(shape).astype(np.float32))

    def us(run):
        times = []
        for _ in range(4):   # the first one warms up
            ms = ctypes.c_float()
            fdx.check(fdx.lib.fdx_timer_start())
            run()
            fdx.check(fdx.lib.fdx_timer_stop(ctypes.byref(ms)))
            times.append(1e3 * ms.value)
        return min(times[1:])

    def compare(name, run, *shape):
        finite, nan = dev(*shape), fdx.DevBuf.from_host(np.full(shape, np.nan, np.float32))
        a, b = us(lambda: fdx.check(run(finite.ptr))), us(lambda: fdx.check(run(nan.ptr)))
        print("%s: finite %.1f us, NaN %.1f us" % (name, a, b), flush=True)
        assert b <= 8 * a, name

    m, n, k = 8192, 2048, 512
    w, w3, out = dev(n, k), dev(128, 3, 3, 128), fdx.DevBuf(4 * m * n)
    fdx.lib.fdx_mha_scratch_bytes.restype = ctypes.c_size_t
    scratch = fdx.DevBuf(fdx.lib.fdx_mha_scratch_bytes(32, 8, 256, 256, 64))
    compare("gemm", lambda x: fdx.lib.fdx_gemm_bias_act_f32(x, ctypes.c_int64(k), w.ptr, ctypes.c_int64(k), m, n, k, ctypes.c_float(1), None, 0,
                                                            None, None, out.ptr, ctypes.c_int64(n), None), m, k)
    compare("convolution", lambda x: fdx.lib.fdx_conv2d_nhwc_f32(x, 16, 28, 28, 128, w3.ptr, None, 128, 3, 3, 1, 1, 1, 1, 1, 1, 28, 28,
                                                                 None, None, out.ptr), 16, 28, 28, 128)
    compare("attention", lambda x: fdx.lib.fdx_mha_prefill_f32(x, x, x, 32, 256, 256, 8, 64, 64, 0, out.ptr, scratch.ptr), 32, 256, 512)


@pytest.mark.parametrize("tile", [23, 24, 28, 223, 10323, 424])
@pytest.mark.parametrize("n,h,w,cin,cout,kh,kw,dil", [
    (2, 9, 7, 32, 64, 3, 3, 1), (3, 14, 14, 64, 132, 3, 3, 1), (1, 28, 56, 32, 64, 3, 3, 1), (9, 7, 7, 96, 260, 3, 3, 1),
    (2, 11, 63, 32, 68, 3, 3, 1),                               # the longest run of pixels: 128 beyond the tile's rows
    (1, 20, 31, 64, 64, 5, 5, 1), (2, 17, 12, 32, 36, 1, 3, 1), (2, 16, 15, 64, 40, 3, 3, 2), (1, 5, 4, 32, 36, 3, 2, 1)])
def test_convolution_halo(fdx, n, h, w, cin, cout, kh, kw, dil, tile):
    """The form that fetches a tile's pixels once for all filter taps: rows of a tile over image borders and images, runs cut at
    both ends of the batch, K ranges that begin inside a channel slab."""
    import torch
    print("halo", n, h, w, cin, cout, kh, kw, dil, tile, flush=True)
    r = np.random.default_rng(zlib.crc32(repr((n, h, w, cin, cout)).encode()))
    x = r.standard_normal((n, h, w, cin)).astype(np.float32)
    wc = (r.standard_normal((cout, kh, kw, cin)) / np.sqrt(kh * kw * cin)).astype(np.float32)
    b, res = r.standard_normal(cout).astype(np.float32), r.standard_normal((n, h, w, cout)).astype(np.float32)
    got, again = forced(fdx, tile, lambda: [fdx.conv2d(x, wc, b, dilation=(dil, dil), padding="same", residual=res) for _ in range(2)])
    eh, ew = (kh - 1) * dil, (kw - 1) * dil
    xp = torch.nn.functional.pad(torch.from_numpy(x).double().permute(0, 3, 1, 2), (ew // 2, ew - ew // 2, eh // 2, eh - eh // 2))
    conv = lambda a, f: torch.nn.functional.conv2d(a, f.permute(0, 3, 1, 2), dilation=dil).permute(0, 2, 3, 1).numpy()
    want, size = conv(xp, torch.from_numpy(wc).double()) + b + res, conv(xp.abs(), torch.from_numpy(wc).double().abs()) + np.abs(b) + np.abs(res)
    k = kh * kw * cin
    assert (np.abs(got - want) <= (k / 16 + 8) * 2.0 ** -23 * size).all()
    assert np.linalg.norm(got - want) <= (1.2e-8 * np.sqrt(k) + 1.2e-7) * np.linalg.norm(want)
    assert np.array_equal(got, again)


@pytest.mark.parametrize("cap", [8, 10])
@pytest.mark.parametrize("tile", [23, 24, 28, 223, 424, 228, 10223, 10323, 10224, 10228])
@pytest.mark.parametrize("kh,kw,cin,dil", [(3, 3, 64, 1), (1, 3, 128, 2), (3, 2, 96, 1)])
def test_convolution_halo_several_tiles_a_workgroup(fdx, kh, kw, cin, dil, tile, cap):
    """A grid of `cap` workgroups: each walks to tiles of another place and of another column block, the next tile's pixels requested
    in front of the epilogue of the one before; the hybrid cuts leave whole tiles and a cut remainder (27 tiles of 128 x 128, 45 of
    128 x 64, 15 of 256 x 128)."""
    import torch
    n, h, w, cout = 3, 20, 19, 260
    bm, bn = {3: (128, 128), 4: (128, 64), 8: (256, 128)}[tile % 10]
    tiles, splits = -(-n * h * w // bm) * -(-cout // bn), tile % 10000 // 100
    assert tiles > cap and tiles % cap != 0 and (splits == 0 or kh * kw * cin // 32 >= 2 * splits)   # the cut is not refused
    print("halo, several tiles", kh, kw, cin, dil, tile, cap, flush=True)
    r = np.random.default_rng(zlib.crc32(repr((kh, kw, cin)).encode()))
    x = r.standard_normal((n, h, w, cin)).astype(np.float32)
    k = kh * kw * cin
    wc = (r.standard_normal((cout, kh, kw, cin)) / np.sqrt(k)).astype(np.float32)
    b, res = r.standard_normal(cout).astype(np.float32), r.standard_normal((n, h, w, cout)).astype(np.float32)
    fdx.lib.fdx_debug_persist_cap(cap)
    try:
        got, again = forced(fdx, tile, lambda: [fdx.conv2d(x, wc, b, dilation=(dil, dil), padding="same", residual=res) for _ in range(2)])
    finally:
        fdx.lib.fdx_debug_persist_cap(0)
    eh, ew = (kh - 1) * dil, (kw - 1) * dil
    xp = torch.nn.functional.pad(torch.from_numpy(x).double().permute(0, 3, 1, 2), (ew // 2, ew - ew // 2, eh // 2, eh - eh // 2))
    conv = lambda a, f: torch.nn.functional.conv2d(a, f.permute(0, 3, 1, 2), dilation=dil).permute(0, 2, 3, 1).numpy()
    want, size = conv(xp, torch.from_numpy(wc).double()) + b + res, conv(xp.abs(), torch.from_numpy(wc).double().abs()) + np.abs(b) + np.abs(res)
    assert (np.abs(got - want) <= (k / 16 + 8) * 2.0 ** -23 * size).all()
    assert np.linalg.norm(got - want) <= (1.2e-8 * np.sqrt(k) + 1.2e-7) * np.linalg.norm(want)
    assert np.array_equal(got, again)
