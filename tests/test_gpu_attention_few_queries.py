"""Attention kernel for few queries in flight (32 queries a workgroup, keys shared out among its waves): numbers of queries
and keys around its blocks, against float64.  Both products and the softmax are float32; a sum of `s` probabilities times
values errs by at most about (s + depth) 2^-24 of the largest value, far above what is seen."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def reference(q, k, v, causal):
    q, k, v = [a.astype(np.float64).transpose(0, 2, 1, 3) for a in (q, k, v)]
    scores = q @ k.transpose(0, 1, 3, 2) / math.sqrt(q.shape[-1])
    if causal:
        t, s = scores.shape[-2:]
        scores = np.where(np.arange(s)[None, :] <= np.arange(t)[:, None] + s - t, scores, -np.inf)
    p = np.exp(scores - scores.max(-1, keepdims=True))
    return (p / p.sum(-1, keepdims=True) @ v).transpose(0, 2, 1, 3)


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("t,s", [(2, 2), (31, 31), (32, 32), (33, 33), (65, 129), (8, 300), (128, 128), (77, 77), (160, 161)])
@pytest.mark.parametrize("causal", [0, 1])
def test_attention(fdx, d, t, s, causal):
    print("attention", d, t, s, causal, flush=True)
    r = np.random.default_rng(81)
    # one sequence (the key-split kernel), and enough of them for the other one
    for batch, heads in ((1, 2), (2, 3), (70, 4)):
        q, k, v = [r.standard_normal((batch, n, heads, d)).astype(np.float32) for n in (t, s, s)]
        got = fdx.mha_prefill(*[a.reshape(batch, a.shape[1], heads * d) for a in (q, k, v)], heads, d, d, causal).reshape(q.shape)
        want = reference(q, k, v, causal)
        assert np.abs(got - want).max() / np.abs(want).max() <= (s + d) * 2.0 ** -24, (batch, heads)
