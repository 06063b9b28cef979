"""KV-cache decode sessions against the oracle's causal definition (row t = the reference's
MultiHeadAttention(query = x[t:t+1], value = x[0:t+1])).  Logits: max|gpu - ref| / max|ref| <= 1e-4;
greedy token ids must be identical wherever the oracle's top-2 logit margin exceeds 1e-3."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-4


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    assert a.shape == b.shape
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-30)


def say(*a):
    print(*a, flush=True)


def oracle_logits(ref, ids):
    """ids [t] -> logits [t, vocab] under causal attention."""
    pos = np.arange(len(ids), dtype=np.float32)
    return ref.predict([np.asarray(ids, np.float32), pos], causal=True)[0]


def margin(row):
    top = np.sort(row)[-2:]
    return top[1] - top[0]


@pytest.mark.parametrize("cfg", [dict(layers=2, d_model=32, heads=4, vocab=97, max_pos=40),
                                 dict(layers=3, d_model=64, heads=2, vocab=211, max_pos=40)])
def test_prefill_then_decode_matches_oracle(fdx, oracle, modelgen, cfg):
    say("session tiny", cfg)
    spec = modelgen.gpt2(seed=31, bias_std=0.1, random_affine=True, std=0.2, **cfg)
    js = modelgen.dumps(spec)
    ref = oracle.OracleModel(js)
    model = fdx.Model(js)
    B, P, N = 3, 7, 6
    r = np.random.default_rng(32)
    prompts = r.integers(0, cfg["vocab"], (B, P))
    sess = fdx.Session(model, B, 32)
    logits, nxt = sess.prefill(prompts)
    seqs = [list(prompts[b]) for b in range(B)]
    for b in range(B):
        want = oracle_logits(ref, seqs[b])[-1]
        assert rel(logits[b], want) <= TOL
        if margin(want) > 1e-3:
            assert nxt[b] == oracle.argmax(want)
    assert sess.length() == P
    # teacher-forced decode steps: feed the oracle's greedy token so both sides see the same history
    for step in range(N):
        feed = []
        for b in range(B):
            feed.append(oracle.argmax(oracle_logits(ref, seqs[b])[-1]))
            seqs[b].append(feed[-1])
        logits, nxt = sess.decode_step(np.array(feed))
        for b in range(B):
            want = oracle_logits(ref, seqs[b])[-1]
            assert rel(logits[b], want) <= TOL, (step, b)
            if margin(want) > 1e-3:
                assert nxt[b] == oracle.argmax(want)
    assert sess.length() == P + N
    # chunked prefill (a second multi-token call on a non-empty cache) equals one long prefill
    sess.reset()
    sess.prefill(prompts[:, :4])
    logits2, _ = sess.prefill(prompts[:, 4:])
    sess.reset()
    logits1, _ = sess.prefill(prompts)
    assert rel(logits2, logits1) <= 1e-5


def test_greedy_loop_equals_stepwise_and_full_recompute(fdx, oracle, modelgen):
    say("session greedy")
    cfg = dict(layers=2, d_model=48, heads=3, vocab=151, max_pos=64)
    js = modelgen.dumps(modelgen.gpt2(seed=33, bias_std=0.1, random_affine=True, std=0.2, **cfg))
    model = fdx.Model(js)
    B, P, N = 4, 9, 12
    prompts = np.random.default_rng(34).integers(0, cfg["vocab"], (B, P))
    sess = fdx.Session(model, B, 64)
    _, first = sess.prefill(prompts)
    tokens, last_logits = sess.decode_greedy(first, N)
    # step-by-step session gives the same tokens
    sess2 = fdx.Session(model, B, 64)
    _, nxt = sess2.prefill(prompts)
    assert np.array_equal(nxt, first)
    cur = first
    for i in range(N):
        logits, nxt = sess2.decode_step(cur)
        assert np.array_equal(nxt, tokens[i])
        cur = nxt
    assert rel(logits, last_logits) <= 1e-6
    # prefix identity on the GPU itself: prefilling the whole generated sequence reproduces the last logits
    full = np.concatenate([prompts, first[:, None], tokens[:-1].T], axis=1)
    sess3 = fdx.Session(model, B, 64)
    logits3, nxt3 = sess3.prefill(full)
    assert rel(logits3, last_logits) <= 1e-5
    # and the oracle agrees on one sequence
    ref = oracle.OracleModel(js)
    want = oracle_logits(ref, full[0])[-1]
    assert rel(last_logits[0], want) <= TOL


def test_session_rejects_non_decoder_models_and_overflow(fdx, modelgen):
    say("session errors")
    cnn = fdx.Model(modelgen.dumps(modelgen.small_cnn()))
    with pytest.raises(fdx.FdxError):
        fdx.Session(cnn, 1, 8)
    js = modelgen.dumps(modelgen.gpt2(seed=35, layers=1, d_model=16, heads=2, vocab=19, max_pos=16))
    sess = fdx.Session(fdx.Model(js), 2, 4)
    sess.prefill(np.zeros((2, 3)))
    sess.decode_step(np.zeros(2))
    with pytest.raises(fdx.FdxError, match="exceeds max_len"):
        sess.decode_step(np.zeros(2))


def test_session_rejects_layers_that_mix_positions(fdx, modelgen):
    """A cached decode step works on one position at a time: LayerNormalization over anything but the depth axis and
    Flatten / Reshape layers (which regroup the (T, depth) sample) are refused when the session is created, instead of
    being computed over one position's depth."""
    say("session: position-mixing layers")
    import copy
    base = modelgen.gpt2(seed=40, layers=1, d_model=16, heads=2, vocab=19, max_pos=16)
    for axis in ([1], [1, 2], [-2]):
        spec = copy.deepcopy(base)
        for layer in spec["architecture"]["config"]["layers"]:
            if layer["name"] == "h0_ln2":
                layer["config"]["axis"] = axis
        with pytest.raises(fdx.FdxError, match="axis other than the last"):
            fdx.Session(fdx.Model(modelgen.dumps(spec), verify=False), 2, 8)
    for cls, cfg in (("Reshape", {"target_shape": [-1, 16]}), ("Flatten", {})):
        b = modelgen.Builder("mix", 41)
        ids, pos = b.input((None,), "ids"), b.input((None,), "positions")
        x = b.add([b.embedding(ids, 19, 16, "wte"), b.embedding(pos, 16, 16, "wpe")], "embed_add")
        h = b.layernorm(x, "ln1", 1e-5)
        h = b.mha(h, h, "attn", 2, 8)
        x = b.add([x, h], "add1")
        x = b._add(cls, "regroup", cfg, [x], x.shape)
        x = b.dense(x, 19, "lm_head")
        model = fdx.Model(modelgen.dumps(b.finish([x])), verify=False)
        with pytest.raises(fdx.FdxError, match="reshapes across positions"):
            fdx.Session(model, 2, 8)
    fdx.Session(fdx.Model(modelgen.dumps(base), verify=False), 2, 8)  # the unmodified decoder is accepted


def test_vocabulary_sized_head_leaves_its_own_argmax(fdx, modelgen):
    """With tens of thousands of logits per row the logits launch strides over the column groups and leaves
    per-workgroup maxima, from which the greedy ids are picked without another pass over the logits: the ids must be
    the first maximum of the logits the same step returns, for batch sizes that fill and do not fill the 16 rows,
    and the captured loop must produce the same tokens as single steps."""
    say("session with a vocabulary-sized head")
    cfg = dict(layers=1, d_model=64, heads=1, vocab=40009, max_pos=32)
    js = modelgen.dumps(modelgen.gpt2(seed=36, bias_std=0.1, random_affine=True, std=0.2, **cfg))
    model = fdx.Model(js)
    for B in (16, 5):
        prompts = np.random.default_rng(37 + B).integers(0, cfg["vocab"], (B, 6))
        sess = fdx.Session(model, B, 32)
        logits, first = sess.prefill(prompts)
        assert np.array_equal(first, np.argmax(logits, -1).astype(first.dtype))
        tokens, last_logits = sess.decode_greedy(first, 7)
        sess2 = fdx.Session(model, B, 32)
        _, cur = sess2.prefill(prompts)
        for i in range(7):
            logits, nxt = sess2.decode_step(cur)
            assert np.array_equal(nxt, np.argmax(logits, -1).astype(nxt.dtype)), (B, i)
            assert np.array_equal(nxt, tokens[i]), (B, i)
            cur = nxt
        assert rel(logits, last_logits) <= 1e-6


def test_attention_with_output_projection_in_one_launch(fdx, oracle, modelgen, monkeypatch):
    """With 64-wide heads the decode step runs attention and the layer's output projection (bias, residual Add) as one
    launch whose per-head partial rows are added in head order by the last workgroup to arrive, when FDX_DECODE_FUSE_PROJ=1
    is set while the session is created (two launches measure slightly faster and are the default).  Both forms against each other, step by step and in the
    captured loop, for a batch that fills the 16 rows and one that does not, and the fused form against the oracle."""
    say("decode attention + output projection, one launch vs two")
    cfg = dict(layers=3, d_model=192, heads=3, vocab=211, max_pos=64)
    js = modelgen.dumps(modelgen.gpt2(seed=38, bias_std=0.1, random_affine=True, std=0.2, **cfg))
    model = fdx.Model(js)
    ref = oracle.OracleModel(js)
    for B in (16, 5):
        P, N = 7, 20
        prompts = np.random.default_rng(39 + B).integers(0, cfg["vocab"], (B, P))
        two = fdx.Session(model, B, 64)
        monkeypatch.setenv("FDX_DECODE_FUSE_PROJ", "1")
        one = fdx.Session(model, B, 64)
        monkeypatch.delenv("FDX_DECODE_FUSE_PROJ")
        _, first = two.prefill(prompts)
        _, first1 = one.prefill(prompts)
        assert np.array_equal(first, first1)
        want_tokens, want_logits = two.decode_greedy(first, N)
        tokens, logits = one.decode_greedy(first1, N)
        assert np.array_equal(tokens, want_tokens)
        assert rel(logits, want_logits) <= 1e-5
        # single steps, twice over the same positions after a reset (the tickets must be back at zero)
        for _ in range(2):
            one.reset()
            two.reset()
            _, cur = one.prefill(prompts)
            two.prefill(prompts)
            for i in range(6):
                la, na = two.decode_step(cur)
                lb, nb = one.decode_step(cur)
                assert np.array_equal(na, nb) and np.array_equal(nb, want_tokens[i])
                assert rel(lb, la) <= 1e-5
                cur = nb
        seq = np.concatenate([prompts[0], first[:1], want_tokens[:5, 0]]).astype(np.float32)
        want = oracle_logits(ref, seq)[-1]
        assert rel(lb[0], want) <= TOL


@pytest.mark.parametrize("B", [16, 7, 6, 5, 1])
def test_embedding_folded_into_its_readers_gives_the_same_tokens(fdx, modelgen, B):
    """The opt-in form of the decode step in which the first projection GEMM and the first residual operand form the
    token + position rows themselves (one launch fewer).  From seven sequences on same sums in the same order, so logits and tokens are
    bit-identical to the default step; up to six the default step's two projections add up in an order of their own, and logits
    agree to the rounding errors of two layers' sums (so do the tokens, unless two logits are that close)."""
    print("decode step with the embedding folded into its readers", B, flush=True)
    js = modelgen.dumps(modelgen.gpt2(seed=61, layers=2, d_model=768, heads=12, vocab=50257, max_pos=128, bias_std=0.1,
                                      random_affine=True))
    model = fdx.Model(js, verify=False)
    P, N = 24, 12
    prompts = np.random.default_rng(62).integers(0, 50257, (B, P))
    outs = []
    for mode in (0, 1):
        fdx.check(fdx.lib.fdx_debug_decode_embed_fold(mode))
        try:
            sess = fdx.Session(model, B, 64)
        finally:
            fdx.check(fdx.lib.fdx_debug_decode_embed_fold(-1))
        _, first = sess.prefill(prompts)
        tokens, logits = sess.decode_greedy(first, N)
        step_logits, step_next = sess.decode_step(tokens[-1])
        outs.append((tokens, logits, step_logits, step_next))
        sess.close()
    for a, b in zip(outs[0], outs[1]):
        if B > 6:
            assert np.array_equal(a, b)
        else:
            assert a.shape == b.shape and rel(a, b) <= 1e-5


def test_greedy_loop_with_the_embedding_in_the_previous_steps_last_launch(fdx, modelgen):
    """Inside a greedy loop over a vocabulary-sized head the token + position embedding of a step rides in the last launch
    of the step before (the loop's first embedding runs ahead of the replays).  The loop, called twice with a single
    step in between, must give the tokens of single steps; a loop that would run past the position table keeps the
    stand-alone embedding launch."""
    say("greedy loop, embedding merged into the arg-max launch")
    cfg = dict(layers=2, d_model=64, heads=2, vocab=40009, max_pos=24)
    js = modelgen.dumps(modelgen.gpt2(seed=63, bias_std=0.1, random_affine=True, std=0.2, **cfg))
    model = fdx.Model(js)
    B = 6
    prompts = np.random.default_rng(64).integers(0, cfg["vocab"], (B, 5))
    loop = fdx.Session(model, B, 32)
    _, first = loop.prefill(prompts)
    part1, _ = loop.decode_greedy(first, 6)            # positions 5 .. 10
    _, mid = loop.decode_step(part1[-1])               # a single step between two loops (position 11)
    part2, last_logits = loop.decode_greedy(mid, 7)    # positions 12 .. 18
    single = fdx.Session(model, B, 32)
    _, cur = single.prefill(prompts)
    want = []
    for i in range(6 + 1 + 7):
        logits, cur_next = single.decode_step(cur)
        want.append(cur_next)
        cur = cur_next
    got = list(part1) + [mid] + list(part2)
    for i, (g, w) in enumerate(zip(got, want)):
        assert np.array_equal(g, w), i
    assert rel(logits, last_logits) <= 1e-6
    # positions 19 .. 23 exist, 24 does not: a loop of 6 from here runs past the table and takes the stand-alone embedding
    # launches, like the single steps (a position without a row contributes zeros in both)
    part3, _ = loop.decode_greedy(part2[-1], 6)
    for i in range(6):
        _, cur = single.decode_step(cur)
        assert np.array_equal(part3[i], cur), i


@pytest.mark.parametrize("heads,d_model,vocab", [(1, 64, 40009), (3, 192, 33000)])
def test_prompts_last_position_runs_through_the_decode_launches(fdx, oracle, modelgen, heads, d_model, vocab):
    """Behind the last attention layer's keys and values a prompt goes on for its last position only, on the decode
    launches: against the oracle, for a first prompt, a continued one and prompts of 1 and 2 tokens, then greedy tokens from
    there; and against a session too long for the decode attention's single pass, which keeps the general launches."""
    say("prompt tail on decode launches", heads, d_model, vocab)
    js = modelgen.dumps(modelgen.gpt2(seed=71, layers=2, d_model=d_model, heads=heads, vocab=vocab, max_pos=96, bias_std=0.1,
                                      random_affine=True, std=0.2))
    model, ref = fdx.Model(js), oracle.OracleModel(js)
    for B in (1, 5, 16):
        ids = np.random.default_rng(72 + B).integers(0, vocab, (B, 50))
        short, long = fdx.Session(model, B, 64), fdx.Session(model, B, 16384)
        for lo, hi in ((0, 37), (37, 38), (38, 40), (40, 50)):
            logits, nxt = short.prefill(ids[:, lo:hi])
            general, _ = long.prefill(ids[:, lo:hi])
            assert np.array_equal(nxt, np.argmax(logits, -1).astype(nxt.dtype)), (B, hi)
            assert rel(logits, general) <= 1e-5, (B, hi)
        assert short.length() == 50
        want = oracle_logits(ref, ids[B - 1].astype(np.float32))[-1]
        assert rel(logits[B - 1], want) <= TOL
        tokens, last = short.decode_greedy(nxt, 3)
        seq = np.concatenate([ids[0], nxt[:1], tokens[:2, 0]]).astype(np.float32)
        assert rel(last[0], oracle_logits(ref, seq)[-1]) <= TOL


@pytest.mark.parametrize("heads,d_model,chunks", [(3, 192, (37, 5, 2)), (12, 768, (130, 63)), (2, 64, (3, 2))])
def test_stacked_projection_writes_the_cache_like_three_launches(fdx, modelgen, heads, d_model, chunks):
    """Sessions of up to 16 sequences project queries, keys and values of a prompt with one GEMM whose column ranges go to
    the query buffer and the two caches; one of 17 sequences takes a launch for each.  Same prompts through both, in ragged
    pieces (tiles that cross sequences, few and many tiles), then greedy tokens, which read every cached row."""
    say("stacked projection", heads, d_model, chunks)
    js = modelgen.dumps(modelgen.gpt2(seed=91, layers=2, d_model=d_model, heads=heads, vocab=307, max_pos=256, bias_std=0.1,
                                      random_affine=True, std=0.1))
    model = fdx.Model(js, verify=False)
    ids = np.random.default_rng(92).integers(0, 307, (17, sum(chunks)))
    wide, stacked, one = fdx.Session(model, 17, 256), fdx.Session(model, 16, 256), fdx.Session(model, 1, 256)
    lo = 0
    for n in chunks:
        want, _ = wide.prefill(ids[:, lo:lo + n])
        got, nxt = stacked.prefill(ids[:16, lo:lo + n])
        single, _ = one.prefill(ids[:1, lo:lo + n])
        assert rel(got, want[:16]) <= 1e-5 and rel(single, want[:1]) <= 1e-5, lo
        lo += n
    cur = np.concatenate([nxt, nxt[:1]])
    want, _ = wide.decode_step(cur)
    got, _ = stacked.decode_step(nxt)
    assert rel(got, want[:16]) <= 1e-5


@pytest.mark.parametrize("step", [6, 9, 11, 12])
def test_a_call_that_fails_half_way_leaves_the_length_alone(fdx, modelgen, step):
    """Prompts and steps move the device's copy of the session length by launches of their own.  Stopped in the last layer, in
    the head or behind the arg-max, they leave the session where it was: what follows equals a session that never failed."""
    say("failing step", step)
    js = modelgen.dumps(modelgen.gpt2(seed=121, layers=2, d_model=192, heads=3, vocab=33000, max_pos=64, bias_std=0.1, std=0.1))
    model = fdx.Model(js, verify=False)
    ids = np.random.default_rng(122).integers(0, 33000, (5, 40))
    hurt, sound = fdx.Session(model, 5, 40), fdx.Session(model, 5, 40)

    def fails(call):
        fdx.check(fdx.lib.fdx_debug_fail_session_step(step))
        try:
            with pytest.raises(fdx.FdxError, match="refused"):
                call()
        finally:
            fdx.check(fdx.lib.fdx_debug_fail_session_step(-1))

    fails(lambda: hurt.prefill(ids[:, :30]))
    assert hurt.length() == 0
    for s in (hurt, sound):
        s.prefill(ids[:, :12])
    fails(lambda: hurt.prefill(ids[:, 12:39]))
    fails(lambda: hurt.decode_step(ids[:, 12]))
    assert hurt.length() == 12
    for s in (hurt, sound):
        s.last = s.decode_step(ids[:, 12])
    assert np.array_equal(hurt.last[0], sound.last[0]) and np.array_equal(hurt.last[1], sound.last[1])
    fails(lambda: hurt.decode_greedy(hurt.last[1], 4))
    a, b = hurt.decode_greedy(hurt.last[1], 4), sound.decode_greedy(sound.last[1], 4)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    assert hurt.length() == sound.length() == 17


@pytest.mark.parametrize("tile", [15, 40, 41, 42, 43, 44])
def test_every_form_of_the_stacked_projection(fdx, modelgen, tile):
    """The stacked projection's forms one by one: three tensors in the first layer, keys and values only in the last, from one
    row block to tiles that cross sequences, against a session of 17 sequences, which takes a launch for each."""
    say("stacked projection", tile)
    js = modelgen.dumps(modelgen.gpt2(seed=131, layers=2, d_model=192, heads=3, vocab=33000, max_pos=128, bias_std=0.1,
                                      random_affine=True, std=0.1))
    model = fdx.Model(js, verify=False)
    ids = np.random.default_rng(132).integers(0, 33000, (17, 90))
    wide = fdx.Session(model, 17, 96)
    some = {B: fdx.Session(model, B, 96) for B in (1, 5, 16)}
    lo = 0
    for n in (2, 3, 16, 63):
        want, _ = wide.prefill(ids[:, lo:lo + n])
        fdx.lib.fdx_debug_force_tile(tile)
        try:
            got = {B: s.prefill(ids[:B, lo:lo + n])[0] for B, s in some.items()}
        finally:
            fdx.lib.fdx_debug_force_tile(-1)
        for B in some:
            assert rel(got[B], want[:B]) <= 1e-5, (B, n)
        lo += n


def test_stacked_projection_timed_and_from_a_table(fdx, modelgen):
    """With timing asked for, the stacked projection's form is timed once per shape and exported; the table comes back in and
    holds for a frozen process."""
    say("stacked projection, timed")
    js = modelgen.dumps(modelgen.gpt2(seed=133, layers=2, d_model=192, heads=3, vocab=307, max_pos=128, bias_std=0.1, std=0.1))
    model = fdx.Model(js, verify=False)
    ids = np.random.default_rng(134).integers(0, 307, (16, 111))
    s = fdx.Session(model, 16, 111)
    want, _ = s.prefill(ids)
    rows = lambda: [r for r in fdx.tuner_export().splitlines() if r.startswith("4 1776 576 192 3 ")]
    assert not rows()
    fdx.tuner_timing(True)
    try:
        s.reset()
        timed, _ = s.prefill(ids)
    finally:
        fdx.tuner_timing(False)
    row, = rows()
    assert int(row.split()[-1]) in (15, 40, 41, 42, 43, 44)
    head = row.rsplit(" ", 1)[0]
    try:
        for choice in (40, 44, 15, 39, 99):  # the last two are no forms: the closed rule
            fdx.tuner_import("%s %d\n" % (head, choice))
            s.reset()
            got, _ = s.prefill(ids)
            assert rel(got, want) <= 1e-5 and rel(timed, want) <= 1e-5, choice
    finally:
        fdx.tuner_import(row + "\n")


LOWEST = np.float32(-3.4028234663852886e38)
HEADS = {
    "NaN among numbers": lambda b: b.__setitem__(slice(3, 40, 9), np.nan),
    "NaN only": lambda b: b.fill(np.nan),
    "-inf only": lambda b: b.fill(-np.inf),
    "the lowest float only": lambda b: b.fill(LOWEST),
    "the lowest float, then NaN": lambda b: (b.fill(LOWEST), b.__setitem__(7, np.nan)),
    "-inf but for one": lambda b: (b.fill(-np.inf), b.__setitem__(17, -1e38)),
    "inf twice": lambda b: b.__setitem__([20, 25], np.inf),
    "0 everywhere": lambda b: b.fill(0),
    "-0 in front of 0": lambda b: (b.fill(-1), b.__setitem__(11, -0.0), b.__setitem__(13, 0.0)),
    "equal largest values": lambda b: b.__setitem__([30, 31, 39], 99),
}


@pytest.mark.parametrize("vocab", [40, 33000])
@pytest.mark.parametrize("head", list(HEADS))
def test_greedy_ids_of_special_logits(fdx, oracle, modelgen, vocab, head):
    """What a prompt, a step and the greedy loop pick follows the reference's scan for the first value above all before it,
    which starts at the lowest float: NaN, -inf and the lowest float never win, id 0 stands for no winner.  With a small head
    the ids come from a pass over the logits, with a large one from the maxima its launch leaves."""
    say("special logits", vocab, head)
    spec = modelgen.gpt2(seed=151, layers=1, d_model=64, heads=1, vocab=vocab, max_pos=32, bias_std=0.1, std=0.1)
    lm = spec["trainable_params"]["lm_head"]
    lm["weights"][:] = 0  # the logits are the bias
    HEADS[head](lm["bias"])
    model = fdx.Model(modelgen.dumps(spec), verify=False)
    want, best = 0, LOWEST
    for i, v in enumerate(lm["bias"]):
        if v > best:
            want, best = i, v
    assert want == oracle.argmax(lm["bias"])
    for B in (1, 5, 17):
        s = fdx.Session(model, B, 32)
        ids = np.random.default_rng(152).integers(0, vocab, (B, 6))
        logits, nxt = s.prefill(ids)
        assert np.array_equal(logits, np.tile(lm["bias"], (B, 1)), equal_nan=True)
        assert nxt.tolist() == [want] * B
        assert s.decode_step(nxt)[1].tolist() == [want] * B
        assert s.decode_greedy(nxt, 3)[0].tolist() == [[want] * B] * 3


def test_prompts_take_the_decode_launches_behind_the_last_cache_rows(fdx, modelgen):
    """Which launches a prompt's last position takes, from the profile: the projections of the decode kernels where the plan
    allows them (its last layer's three and the head, one attention launch and the arg-max of the head's maxima), none of them
    in a session that is too long for the decode attention."""
    say("launches of a prompt")
    c = fdx.ctypes
    model = fdx.Model(modelgen.dumps(modelgen.gpt2(seed=161, layers=2, d_model=192, heads=3, vocab=33000, max_pos=64, std=0.1)), verify=False)

    def families(max_len):
        s = fdx.Session(model, 4, max_len)
        fdx.check(fdx.lib.fdx_profile_enable(1))
        try:
            fdx.check(fdx.lib.fdx_profile_reset())
            s.prefill(np.arange(4 * 9).reshape(4, 9))
            fdx.sync()
            seen, i = {}, 0
            name, n, ms, fl, by = c.create_string_buffer(128), c.c_uint64(), c.c_double(), c.c_double(), c.c_double()
            while fdx.lib.fdx_profile_get(i, name, 128, c.byref(n), c.byref(ms), c.byref(fl), c.byref(by)) == 0:
                seen[name.value.decode()] = n.value
                i += 1
        finally:
            fdx.check(fdx.lib.fdx_profile_enable(0))
        return seen

    short, long = families(64), families(16384)
    print(short, long, flush=True)
    assert short.get("dense_rows_f32") == 5 and short.get("mha_decode_f32") == 1 and short.get("mha_flash_f32") == 1
    assert "dense_rows_f32" not in long and "mha_decode_f32" not in long and long.get("mha_flash_f32") == 2
