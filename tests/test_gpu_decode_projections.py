"""Projections of decode steps over packed filters: the forms that the sequences' number and the K range of a workgroup choose
(rows loaded directly or through LDS, 6, 8 or 24 slabs a wave or a loop over them, K whole or cut with the exchange inside an
XCD or through tickets), at the edges of their ranges, against the oracle and against the same tokens in sessions of other
sizes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-4  # as for the other session tests


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    assert a.shape == b.shape
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-30)


@pytest.mark.parametrize("d_model,heads,ffn,vocab", [
    (256, 4, 1024, 311),     # 256: direct; 1024 floats in one workgroup: eight slabs a wave
    (1024, 16, 4096, 300),   # 1024 under a LayerNormalization; 4096 cut into four ranges of 1024, 64 column groups
    (432, 6, 1728, 307),     # the last width whose rows are loaded directly; ranges of 432
    (448, 7, 1800, 307),     # the first through LDS; 1800 in ranges of 464, the last one short, with waves of one slab and none
    (400, 5, 1600, 290),     # ranges of 400, 25 column groups: the ranges meet through tickets
    (1280, 20, 1300, 305),   # projections without a folded LayerNormalization, cut in two
    (64, 2, 25600, 97),      # eight ranges of 3200: a loop over chunks
    (1040, 13, 64, 33000),   # a head of 1040 floats, too many column groups to cut: 24 slabs a wave
])
def test_decode_projections(fdx, oracle, modelgen, d_model, heads, ffn, vocab):
    js = modelgen.dumps(modelgen.gpt2(seed=141, layers=1, d_model=d_model, heads=heads, vocab=vocab, max_pos=16, ffn=ffn, bias_std=0.1,
                                      random_affine=True, std=0.1))
    ref, model = oracle.OracleModel(js), fdx.Model(js)
    ids = np.random.default_rng(142).integers(0, vocab, (16, 7))
    want = {b: ref.predict([ids[b].astype(np.float32), np.arange(7, dtype=np.float32)], causal=True)[0] for b in (0, 7, 15)}
    steps = {}
    for B in (1, 7, 8, 11, 16):
        print("decode projections", d_model, ffn, vocab, B, flush=True)
        s = fdx.Session(model, B, 16)
        s.prefill(ids[:B, :5])
        steps[B] = [s.decode_step(ids[:B, t])[0] for t in (5, 6)]
        again = s.decode_greedy(np.argmax(steps[B][1], -1), 2)
        s.reset()
        s.prefill(ids[:B, :5])
        for t in (5, 6):
            assert np.array_equal(s.decode_step(ids[:B, t])[0], steps[B][t - 5])  # partial tiles are added in a fixed order
        twice = s.decode_greedy(np.argmax(steps[B][1], -1), 2)
        assert np.array_equal(again[0], twice[0]) and np.array_equal(again[1], twice[1])
        for b in want:
            if b < B:
                for t in (5, 6):
                    assert rel(steps[B][t - 5][b], want[b][t]) <= TOL, (B, b, t)
    for B in (1, 7, 8, 11):
        for t in (0, 1):
            assert rel(steps[B][t], steps[16][t][:B]) <= 1e-5, (B, t)
