"""Attention with many queries at depths 32 and 64: both products on bf16 matrix instructions with operands split exactly in
three.  Against 64 bits.  Scores are sums of D products rounded about D / 16 + 8 times at most at their magnitudes' sum S
(about 0.64 sqrt(D) here after scaling), which is the relative error of a probability; the output sums add as much again:
2 (D / 16 + 8) 2^-24 0.64 sqrt(D) = 7e-6 at depth 64 if all roundings went the same way; they average out, and 1e-6 in the
2-norm leaves a factor of three over what is seen."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def reference(q, k, v, heads, causal):
    b, t, s = q.shape[0], q.shape[1], k.shape[1]
    q, k, v = (x.astype(np.float64).reshape(b, x.shape[1], heads, -1).transpose(0, 2, 1, 3) for x in (q, k, v))
    x = q @ k.transpose(0, 1, 3, 2) / np.sqrt(q.shape[-1])
    if causal:
        x = np.where(np.arange(s)[None, :] <= np.arange(t)[:, None] + s - t, x, -np.inf)
    x = np.exp(x - x.max(-1, keepdims=True))
    return (x / x.sum(-1, keepdims=True) @ v).transpose(0, 2, 1, 3).reshape(b, t, -1)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,t,s,heads,d", [(16, 128, 128, 8, 64), (14, 65, 65, 16, 64), (16, 257, 300, 4, 64), (40, 129, 191, 3, 32),
                                           (32, 33, 64, 12, 32), (64, 96, 97, 3, 64), (12, 511, 511, 4, 32)])
def test_against_64_bits(fdx, b, t, s, heads, d, causal):
    print("attention split", b, t, s, heads, d, causal, flush=True)
    assert (t + 31) // 32 * b * heads > 448   # below that the kernel for few queries takes the launch
    r = np.random.default_rng(b * t + d)
    q, k, v = (r.standard_normal((b, n, heads * d)).astype(np.float32) for n in (t, s, s))
    got, want = fdx.mha_prefill(q, k, v, heads, d, d, causal=causal), reference(q, k, v, heads, causal)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    print("relative error %.2e" % err, flush=True)
    assert err <= 1e-6
    # scores of a few hundred: the running maximum moves from tile to tile
    got, want = fdx.mha_prefill(q * 40, k, v, heads, d, d, causal=causal), reference(q * 40, k, v, heads, causal)
    assert np.linalg.norm(got - want) / np.linalg.norm(want) <= 4e-5


@pytest.mark.parametrize("d", [32, 64])
def test_tiny_operands(fdx, d):
    """Keys, queries, values and probabilities whose last bits lie below bf16's range: the bound of ordinary operands."""
    b, t, heads = 16, 128, 8
    r = np.random.default_rng(2)
    q, k, v = (r.standard_normal((b, t, heads * d)).astype(np.float32) for _ in range(3))
    for eq, ek, ev in ((120, -122, 0), (-122, 120, 0), (0, 0, -122), (127 - 8, -137, 0)):
        print("attention split tiny", d, eq, ek, ev, flush=True)
        x = [np.ldexp(a.astype(np.float64), e).astype(np.float32) for a, e in ((q, eq), (k, ek), (v, ev))]
        got, want = fdx.mha_prefill(*x, heads, d, d), reference(*x, heads, False)
        got = got.astype(np.float64)
        assert np.linalg.norm(got - want) / np.linalg.norm(want) <= 1e-6, (d, eq, ek, ev)
    # One key with probability 1 and value 0, the others' probabilities e^-84 and below, which make the whole output.  An exponent
    # of 84 log2(e) = 121 is held to 2^-18 in fp32: 4e-6 of a probability.
    q, k, v = np.zeros_like(q), np.zeros_like(k), v * np.float32(2.0 ** 60)
    q[:, :, ::d], k[:, 1:, ::d], v[:, 0] = np.sqrt(d), -84 - r.random((b, t - 1, heads)), 0
    got, want = fdx.mha_prefill(q, k, v, heads, d, d), reference(q, k, v, heads, False)
    assert np.linalg.norm(got - want) / np.linalg.norm(want) <= 8e-6


def test_infinities_and_nan(fdx):
    """Operands that the split cannot hold: the queries they reach get the values of plain sums, the others stay as they are."""
    print("attention split special", flush=True)
    b, t, heads, d = 16, 130, 4, 64
    r = np.random.default_rng(1)
    q, k, v = (r.standard_normal((b, t, heads * d)).astype(np.float32) for _ in range(3))
    clean = fdx.mha_prefill(q, k, v, heads, d, d)
    q[1, 5, 0] = np.nan              # one query of head 0
    k[2, 7, 64:128] = 0
    k[2, 7, 64] = -np.inf            # head 1: scores of minus or plus infinity by the sign of the query's first component
    v[3, 9, 128] = np.inf            # head 2: one output column
    q[4, 6, 192] = 3.4e38            # head 3: rounds up to an infinite bf16, its scores are of ordinary size
    k[4, :, 192] *= np.float32(1e-38)
    got = fdx.mha_prefill(q, k, v, heads, d, d)
    with np.errstate(all="ignore"):
        want = reference(q, k, v, heads, False)
    same = np.ones((b, t, heads * d), bool)
    same[1, 5, :64] = same[2, :, 64:128] = same[3, :, 128:192] = same[4, :, 192:] = False
    assert np.array_equal(got[same], clean[same])
    assert np.isnan(got[1, 5, :64]).all()
    neg = q[2, :, 64] > 0            # score -Inf: that key drops out
    assert np.allclose(got[2, neg, 64:128], want[2, neg, 64:128], rtol=1e-4, atol=1e-5) and np.isnan(got[2, ~neg, 64:128]).all()
    assert np.isinf(got[3, :, 128]).all() and np.allclose(got[3, :, 129:192], clean[3, :, 129:192], rtol=1e-4, atol=1e-5)
    assert np.allclose(got[4, :, 192:], want[4, :, 192:], rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("d", [32, 64])
def test_infinities_under_the_causal_mask(fdx, d):
    """A query takes no part of a key that it may not see, whatever the key and its value hold; in a wave of 32 queries any number
    may be taken again, four at a time."""
    print("attention split causal special", d, flush=True)
    b, t, heads = 16, 150, 8         # enough queries for the kernel with split operands
    r = np.random.default_rng(3)
    q, k, v = (r.standard_normal((b, t, heads * d)).astype(np.float32) for _ in range(3))
    clean = fdx.mha_prefill(q, k, v, heads, d, d, causal=True)
    k[0, 71, 0] = np.nan             # sequence 0, head 0: queries from 71 on are NaN
    v[1, 100, 1] = np.inf            # sequence 1, head 0, depth 1: infinite from 100 on
    q[2, [3, 40, 41, 77, 78, 79, 80, 149], 0] = np.nan
    got = fdx.mha_prefill(q, k, v, heads, d, d, causal=True)
    same = np.ones((b, t, heads * d), bool)
    same[0, 71:, :d] = same[1, 100:, :d] = same[2, [3, 40, 41, 77, 78, 79, 80, 149], :d] = False
    assert np.isnan(got[0, 71:, :d]).all() and np.isnan(got[2, [3, 40, 41, 77, 78, 79, 80, 149], :d]).all()
    assert np.isposinf(got[1, 100:, 1]).all()
    rest = [0] + list(range(2, d))
    assert np.allclose(got[1, 100:, rest], clean[1, 100:, rest], rtol=1e-4, atol=1e-5)
    # a tile of 64 keys holds values that some of its queries may not see: those are taken again, to fp32 sums in another order
    assert np.allclose(got[same], clean[same], rtol=1e-4, atol=1e-5)
    assert np.array_equal(got[3:], clean[3:])
