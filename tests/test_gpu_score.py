"""Perplexity scoring on the device kernels (qh_score): the reference's perplexity page scores a
passage one token at a time through the cache and takes -log softmax at the true next token
(web/perplexity.html:146-170). Here the positions run in one batched pass with the bits of one
decode step after another (int8/int4 codes read by the kernels, not an f16 round trip; up to three
as steps), and the log-softmax runs on the device in f64.

Checks, per weight format and numerics mode:
  - each NLL equals the oracle's expression (oracle/oracle.c `or_nll`) applied to the logits the
    same step returns through forward() (same kernels, so the same f32 logits): 1e-12;
  - against the CPU oracle's own logits for the same fed tokens: within what the logit tolerance
    allows (|dNLL| <= 2 x 1e-4 x max|logit|, test/model.test.js:40), exactly (1e-11) for the exact
    numerics, whose logits equal the oracle's;
  - the cache holds the same K/V rows as the forward() run."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

LOGIT_REL = 1e-4      # test/model.test.js:40


def tiny(hip):
    return hip.ModelConfig(hidden=128, intermediate=256, layers=2, heads=2, kv_heads=1, vocab=1000)


@pytest.mark.parametrize("numerics", ["fast", "exact"])
@pytest.mark.parametrize("scheme", ["f16", "int8", "int4"])
def test_score_matches_step_logits_and_the_oracle(ctx, hip, scheme, numerics):
    cfg = tiny(hip)
    ckpt = hip.synthesize_checkpoint(cfg, seed=31)
    lm = "f16" if scheme == "f16" else "int8"
    model = hip.GpuModel.load(ctx, hip.device_tensors(ckpt, cfg, scheme, 128, lm), cfg, maxPositions=128,
                              numerics=numerics)
    ids = hip.synth_tokens(31, "score.ids", cfg.vocab, 30)
    scored = model.newCache(64)
    nll = model.score(ids, scored)
    assert nll.shape == (29,) and scored.length == 29

    stepped = model.newCache(64)
    oracle = O.OracleModel(cfg, ckpt, scheme=scheme, group=128, lm_head=lm, kv_f16=True)
    oc = oracle.new_cache(64)
    worst = 0.0
    for t in range(29):
        out = model.forward_tokens([ids[t]], stepped)
        assert nll[t] == pytest.approx(O.nll(out["logits"], ids[t + 1]), rel=1e-12, abs=1e-12)
        ol = oracle.forward([ids[t]], oc)
        diff = abs(nll[t] - O.nll(ol, ids[t + 1]))
        bound = 1e-11 if numerics == "exact" else 2 * LOGIT_REL * float(np.max(np.abs(ol)))
        assert diff <= bound, (t, diff, bound)
        worst = max(worst, diff)
    ppl = float(np.exp(nll.mean()))
    print(f"{scheme}-{numerics}: perplexity {ppl:.4f} over 29 positions, worst |dNLL| vs the oracle {worst:.2e}")
    for L in range(cfg.layers):
        a, b = scored.present(L), stepped.present(L)
        np.testing.assert_array_equal(a["key"].view(np.uint32), b["key"].view(np.uint32))
        np.testing.assert_array_equal(a["value"].view(np.uint32), b["value"].view(np.uint32))
    scored.destroy()
    stepped.destroy()
    model.destroy()


def test_score_continues_from_a_prompt(ctx, hip):
    """Scoring after a batched prefill scores the later tokens with the full left context."""
    cfg = tiny(hip)
    ckpt = hip.synthesize_checkpoint(cfg, seed=32)
    model = hip.GpuModel.load(ctx, hip.device_tensors(ckpt, cfg, "int4", 128, "int8"), cfg, maxPositions=128)
    ids = hip.synth_tokens(32, "score.context", cfg.vocab, 40)
    a = model.newCache(64)
    whole = model.score(ids, a)
    b = model.newCache(64)
    model.forward_tokens(ids[:15], b, wantLogits=False)   # positions 0..14 in one batched pass
    tail = model.score(ids[15:], b)                        # feeds ids[15..38], scores ids[16..39]
    assert tail.shape == (24,) and b.length == 15 + 24
    # the batched prefill equals one-position steps bit for bit, so the scores agree exactly
    np.testing.assert_array_equal(whole[15:], tail)
    a.destroy()
    b.destroy()
    model.destroy()


def test_score_errors(ctx, hip):
    cfg = tiny(hip)
    ckpt = hip.synthesize_checkpoint(cfg, seed=33)
    model = hip.GpuModel.load(ctx, hip.device_tensors(ckpt, cfg, "int8", 128, "int8"), cfg, maxPositions=64)
    c = model.newCache(8)
    with pytest.raises(hip.QwenHipError, match="at least two tokens"):
        model.score([1], c)
    with pytest.raises(hip.RangeError, match="outside the vocabulary"):
        model.score([1, cfg.vocab], c)
    with pytest.raises(hip.RangeError, match="cannot add"):
        model.score(list(range(12)), c)
    assert c.length == 0
    c.destroy()
    model.destroy()


@pytest.fixture(scope="module", params=["fast", "exact"])
def stepped(request, ctx, hip):
    """A tiny model, 636 ids, and what one-token forwards of them give: logits, K/V rows."""
    numerics = request.param
    cfg = tiny(hip)
    model = hip.GpuModel.load(ctx, hip.device_tensors(hip.synthesize_checkpoint(cfg, seed=34), cfg, "int8", 128, "int8"),
                              cfg, maxPositions=700, numerics=numerics)
    ids = hip.synth_tokens(34, "score.long", cfg.vocab, 637)
    c = model.newCache(700)
    logits = np.empty((636, cfg.vocab), np.float32)
    for t in range(636):
        logits[t] = model.forward_tokens(ids[t:t + 1], c)["logits"]
    kv = [c.present(L) for L in range(cfg.layers)]
    yield model, cfg, ids, logits, kv
    c.destroy()
    model.destroy()


@pytest.mark.parametrize("past,total", [
    (0, 1), (0, 2), (0, 3), (0, 4), (0, 64),
    (0, 65),                    # a last head slice of one row
    (0, 128), (0, 513),         # a second chunk of one position
    (0, 600),                   # a second chunk with two head slices
    (35, 1), (35, 2), (35, 130), (35, 601),
])
def test_score_of_every_slice_equals_steps(hip, stepped, past, total):
    """Every position's score, wherever it falls among chunks of 512 positions and slices of 64 head
    rows: the expression over the steps' own logits (the sum's spans are regrouped: 1e-12), the
    steps' K/V rows, and a cache that goes on as after the steps."""
    model, cfg, ids, logits, kv = stepped
    c = model.newCache(700)
    if past:
        model.forward_tokens(ids[:past], c, wantLogits=False)
    nll = model.score(ids[past:past + total + 1], c)
    assert nll.shape == (total,) and c.length == past + total
    for t in range(total):
        assert nll[t] == pytest.approx(O.nll(logits[past + t], ids[past + t + 1]), rel=1e-12, abs=1e-12), t
    for L in range(cfg.layers):
        p = c.present(L)
        for name in ("key", "value"):
            np.testing.assert_array_equal(p[name].view(np.uint32), kv[L][name][:, :past + total].view(np.uint32))
    last = logits[past + total - 1]
    np.testing.assert_array_equal(c.vector("logits").view(np.uint32), last.view(np.uint32))
    b = model.newCache(700)
    for i in range(0, past + total, 300):
        model.forward_tokens(ids[i:min(i + 300, past + total)], b, wantLogits=False)
    first = int(np.argmax(last))
    assert list(model.decode(c, first, 5)) == list(model.decode(b, first, 5))
    np.testing.assert_array_equal(c.vector("logits").view(np.uint32), b.vector("logits").view(np.uint32))
    b.destroy()
    c.destroy()


def test_score_between_forwards_of_every_mode(hip, stepped):
    """Scores and forwards in turn under each matmul mode share one workspace: results stay those of
    the mode alone."""
    model, cfg, ids, logits, _ = stepped
    want = {}
    for mode in ("batched", "matvec", "mfma"):
        model.set_matmul(mode)
        c = model.newCache(64)
        want[mode] = model.forward_tokens(ids[:40], c)["logits"]
        c.destroy()
    c = model.newCache(64)
    for turn in range(3):
        for mode in ("mfma", "batched", "matvec", "mfma"):
            model.set_matmul(mode)
            c.length = 0
            np.testing.assert_array_equal(model.forward_tokens(ids[:40], c)["logits"].view(np.uint32),
                                          want[mode].view(np.uint32), err_msg=f"{mode}, turn {turn}")
            c.length = 0
            nll = model.score(ids[:21], c)
            for t in range(20):
                assert nll[t] == pytest.approx(O.nll(logits[t], ids[t + 1]), rel=1e-12, abs=1e-12)
    model.set_matmul("batched")
    c.destroy()


@pytest.mark.parametrize("numerics", ["fast", "exact"])
@pytest.mark.parametrize("case", ["span of -inf", "NaN", "+inf", "all -inf"])
def test_score_of_special_logits(ctx, hip, case, numerics):
    """Logits with a whole span of -inf, a NaN, a +inf or nothing but -inf: what the expression gives
    over the whole row, batched and step by step."""
    cfg = tiny(hip)
    ckpt = hip.synthesize_checkpoint(cfg, seed=35)
    embed = ckpt["model.embed_tokens.weight"]
    embed[:, 0] = 0x42C8                        # 100: dimension 0 stays positive in every row
    t = hip.device_tensors(ckpt, cfg, "int8", 128, "f16")
    fmt, rows, cols, group, head, s, z = t["lm_head.weight"]
    head = head.copy()
    only0 = np.zeros(cols, np.uint16)
    if case == "span of -inf":
        only0[0] = 0xFC00                       # -inf
        head[250:375] = only0                   # one eighth of the 1000
    elif case == "NaN":
        head[700, 3] = 0x7E00
    elif case == "+inf":
        only0[0] = 0x7C00
        head[999] = only0
    else:
        only0[0] = 0xFC00
        head[:] = only0
    t["lm_head.weight"] = (fmt, rows, cols, group, head, s, z)
    model = hip.GpuModel.load(ctx, t, cfg, maxPositions=64, numerics=numerics)
    ids = np.array([5, 17, 300, 800, 999, 251, 42, 374, 375, 249], np.int32)
    c, b = model.newCache(64), model.newCache(64)
    nll = model.score(ids, c)
    for i in range(9):
        row = model.forward_tokens(ids[i:i + 1], b)["logits"]
        assert not np.isfinite(row).all()
        want = O.nll(row, ids[i + 1])
        b.length = i
        one = model.score(ids[i:i + 2], b)[0]
        for got in (nll[i], one):
            np.testing.assert_allclose(got, want, rtol=1e-12, err_msg=f"position {i}")
    c.destroy()
    b.destroy()
    model.destroy()
