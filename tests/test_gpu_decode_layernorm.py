"""LayerNormalization inside the decode kernels on rows whose mean is large against their deviation, against float64.

The filters' rows add up to zero, so that what is left of a rounded mean meets nothing: the products of centred rows err by
their own roundings only, while products of the raw rows would carry roundings of the mean's size."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def zero_sum(w, axis):
    return (w - w.mean(axis, keepdims=True, dtype=np.float64)).astype(np.float32)


@pytest.mark.parametrize("m,k,n", [(16, 768, 2304), (3, 64, 100), (16, 768, 50257), (7, 1024, 40), (16, 100, 64), (16, 1024, 40000)])
@pytest.mark.parametrize("ratio", [10, 1000])
def test_layernorm_dense_rows_far_from_zero(fdx, m, k, n, ratio):
    print("layernorm dense rows far from zero", m, k, n, ratio, flush=True)
    r = np.random.default_rng(111)
    x = (r.standard_normal((m, k)) + ratio).astype(np.float32)
    w = np.repeat(r.standard_normal((n, k // 2)) / np.sqrt(k), 2, axis=1).astype(np.float32)
    w[:, 1::2] *= -1  # pairs: the rows add up to zero exactly
    b = r.standard_normal(n).astype(np.float32)
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    d = (x64 - x64.mean(-1, keepdims=True)) / np.sqrt(x64.var(-1, keepdims=True) + 1e-5)
    want = d @ w64.T + b
    dx, dw, db = (fdx.DevBuf.from_host(a) for a in (x, w, b))
    wf, ws, bf, out = fdx.DevBuf(4 * n * k), fdx.DevBuf(4 * n), fdx.DevBuf(4 * n), fdx.DevBuf(4 * m * n)
    fdx.check(fdx.lib.fdx_fold_layernorm_f32(None, None, fdx._dp(dw), fdx._dp(db), n, k, fdx._dp(wf), fdx._dp(ws), fdx._dp(bf)))
    fdx.check(fdx.lib.fdx_layernorm_dense_rows_f32(fdx._dp(dx), m, k, fdx.ctypes.c_float(1e-5), fdx._dp(wf), fdx._dp(ws),
                                                   fdx._dp(bf), n, None, None, fdx._dp(out)))
    # a product is a chain of k / 32 accumulations in each of eight waves (four products at a time), then eight partial
    # sums; centring, scaling and bias add a rounding each.  The mean itself is off by up to about 40 roundings of its
    # size, which the deviations keep as a shift: it meets the zero row sums, but moves the variance by its square.
    eps = 2.0 ** -24
    bound = (k / 32 + 4 + 8 + 4) * eps * (np.abs(d) @ np.abs(w64).T).max() + 0.5 * (40 * eps * ratio) ** 2 * np.abs(want).max()
    assert np.abs(out.to_host((m, n)) - want).max() <= bound


def erf(x):
    return np.vectorize(math.erf)(x)


def logits64(p, heads, ids):
    """Last position's logits of a one-layer decoder of modelgen.gpt2, in float64."""
    f = lambda a: np.asarray(a, np.float64)
    ln = lambda a: (a - a.mean(-1, keepdims=True)) / np.sqrt(a.var(-1, keepdims=True) + 1e-5)
    x = f(p["wte"]["weights"])[ids] + f(p["wpe"]["weights"])[:len(ids)]
    wq, bq, wk, bk, wv, bv, wo, bo = [f(a) for a in p["h0_attn"]["weights"]]
    h = ln(x)
    q, k, v = [np.einsum("td,dhe->the", h, w) + b for w, b in ((wq, bq), (wk, bk), (wv, bv))]
    s = np.einsum("he,the->ht", q[-1], k) / math.sqrt(q.shape[-1])
    s = np.exp(s - s.max(-1, keepdims=True))
    o = np.einsum("ht,the->he", s / s.sum(-1, keepdims=True), v)
    y = x[-1] + np.einsum("he,hed->d", o, wo) + bo
    g = ln(y) @ f(p["h0_fc"]["weights"]) + f(p["h0_fc"]["bias"])
    y = y + (0.5 * g * (1 + erf(g / math.sqrt(2)))) @ f(p["h0_proj"]["weights"]) + f(p["h0_proj"]["bias"])
    return ln(y) @ f(p["lm_head"]["weights"]) + f(p["lm_head"]["bias"])


def test_prompts_and_steps_far_from_zero(fdx, modelgen):
    """A decoder whose residual stream has a mean of 100 deviations: the last position of a prompt and a decode step on the
    decode launches (filters as they are for one sequence, packed for more; rows loaded directly for seven, through LDS for sixteen) are about as close to
    float64 as the launch-by-launch path of a session too long for them, which normalises in a launch of its own."""
    heads, d_model, vocab = 8, 512, 33000
    spec = modelgen.gpt2(seed=112, layers=1, d_model=d_model, heads=heads, vocab=vocab, max_pos=32, bias_std=0.02)
    p = spec["trainable_params"]
    p["wte"]["weights"] += np.float32(100 * 0.02 * math.sqrt(2))
    for i in (0, 2, 4):
        p["h0_attn"]["weights"][i] = zero_sum(p["h0_attn"]["weights"][i], 0)
    for name in ("h0_fc", "lm_head"):
        p[name]["weights"] = zero_sum(p[name]["weights"], 0)
    model = fdx.Model(modelgen.dumps(spec), verify=False)
    for B in (1, 7, 16):
        print("prompt far from zero", B, flush=True)
        ids = np.random.default_rng(113).integers(0, vocab, (B, 12))
        want = [np.stack([logits64(p, heads, ids[b, :t]) for b in range(B)]) for t in (11, 12)]
        got = []
        for max_len in (64, 16384):  # the longer one keeps the general launches for its prompts
            s = fdx.Session(model, B, max_len)
            got.append([s.prefill(ids[:, :11])[0], s.prefill(ids[:, 11:])[0] if max_len > 64 else s.decode_step(ids[:, 11])[0]])
        for step in range(2):
            err = [np.abs(g[step] - want[step]).max() / np.abs(want[step]).max() for g in got]
            print("errors", err, flush=True)
            # both carry the same two roundings of the stream (100 deviations x 2^-24 each); which way they fall differs
            assert err[0] <= 2 * err[1] + 1e-6, (B, step, err)
