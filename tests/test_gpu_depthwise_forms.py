"""Depthwise 3x3, stride 1, on both sides of the line between the row-by-row and the sliding-window form (750000 output
vectors of four channels, or as many in fours of columns where a row has 320 items), ragged widths and heights, against the
oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w,c", [(1, 1, 1, 4), (1, 5, 3, 8), (2, 7, 9, 20), (3, 21, 21, 192), (1, 33, 6, 36), (2, 250, 375, 16),
                                     (2, 251, 375, 16), (47, 28, 29, 80), (48, 28, 29, 80), (77, 14, 14, 200)])
@pytest.mark.parametrize("padding", ["same", "valid"])
def test_dwconv3x3(fdx, oracle, n, h, w, c, padding):
    if padding == "valid" and (h < 3 or w < 3):
        pytest.skip("no output")
    print("dwconv 3x3", n, h, w, c, padding, flush=True)
    r = np.random.default_rng(101)
    x = r.standard_normal((n, h, w, c)).astype(np.float32)
    wj = r.standard_normal((c, 3, 3)).astype(np.float32)
    b = r.standard_normal(c).astype(np.float32)
    got = fdx.dwconv2d(x, wj, b, (1, 1), (1, 1), padding)
    pick = sorted({0, n - 1})
    want = np.stack([oracle.depthwise_conv2d(x[i], wj, b, 3, 3, (1, 1), (1, 1), padding) for i in pick])
    # nine products and a bias in another order: at most 10 roundings of 2^-24 on each side, of sums below 4 times the output
    assert np.abs(got[pick] - want).max() / np.abs(want).max() <= 4 * 20 * 2.0 ** -24


@pytest.mark.parametrize("n,h,w,c,padding", [
    # sliding window with row tiles of 4 (fewer than 65536 items in taller ones): column tiles of 7 and of 8, extents that end
    # inside a tile, both paddings
    (64, 14, 14, 256, "same"), (64, 7, 7, 960, "same"), (62, 9, 11, 512, "same"), (16, 21, 16, 768, "valid"), (20, 21, 22, 512, "valid"),
    (24, 16, 16, 640, "valid"),
    # below 750000 vectors but not in fours: rows of 660, 525, 320 items, and of 315, which stay row by row
    (8, 38, 13, 660, "same"), (40, 10, 10, 700, "same"), (59, 10, 13, 320, "same"), (59, 10, 9, 420, "same"), (8, 40, 15, 660, "valid"),
])
def test_dwconv3x3_sliding_window_without_bias_and_with_relu6(fdx, oracle, n, h, w, c, padding):
    print("dwconv 3x3 sliding window", n, h, w, c, padding, flush=True)
    r = np.random.default_rng(102)
    x = r.standard_normal((n, h, w, c)).astype(np.float32)
    wj = r.standard_normal((c, 3, 3)).astype(np.float32)
    b = r.standard_normal(c).astype(np.float32)
    pick = sorted({0, n // 2, n - 1})
    raw = np.stack([oracle.depthwise_conv2d(x[i], wj, None, 3, 3, (1, 1), (1, 1), padding) for i in pick])
    # as above; a ReLU6 passes errors on
    bound = 4 * 20 * 2.0 ** -24 * np.abs(raw).max()
    plain = fdx.dwconv2d(x, wj, None, (1, 1), (1, 1), padding)[pick]
    assert np.abs(plain - raw).max() <= bound
    got = fdx.dwconv2d(x, wj, b, (1, 1), (1, 1), padding, act=fdx.relu_act(6.0))[pick]
    assert np.abs(got - np.clip(raw + b, 0, 6)).max() <= bound + 2.0 ** -23 * np.abs(raw + b).max()
