"""Depthwise 3x3, stride 1, on both sides of the line between the row-by-row and the sliding-window form (750000 output
vectors of four channels), ragged widths and heights, against the oracle."""
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
