"""Exact attention of a prompt by tiles of 16 queries (csrc/ops.hip k_attn_tile): every query
equals its own one-query call bit for bit, at the edges of the tiles and of the score rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seq,past,heads,kv_heads", [
    (16, 0, 14, 2), (17, 0, 2, 1), (31, 5, 14, 2), (40, 472, 14, 2),   # the last fills 512 positions
    (16, 497, 4, 4), (48, 976, 8, 2), (20, 2028, 2, 1), (130, 3, 4, 2),
])
def test_query_tiles_equal_single_queries_bitwise(ctx, hip, seq, past, heads, kv_heads):
    total = past + seq
    rng = np.random.default_rng(seq * 1000 + past)
    vs = (total + 63) // 64 * 64
    k = rng.standard_normal((kv_heads, total, 64)).astype(np.float16)
    v = np.zeros((kv_heads, 64, vs), np.float16)
    v[:, :, :total] = rng.standard_normal((kv_heads, 64, total))
    v[0, 3, total - 1] = np.inf      # seen by the last query alone: the others must not meet it
    k[0, total - 2] = np.nan         # likewise: the last two queries' softmax is NaN, no other's
    q = rng.standard_normal((seq, heads * 64)).astype(np.float32)
    kc, vc, dq = ctx.upload(k), ctx.upload(v), ctx.upload(q)
    out, one = ctx.empty(q.nbytes), ctx.empty(heads * 64 * 4)
    ctx.attention(dq, kc, vc, total, out, seq, past, heads, kv_heads, kind="exact")
    got = out.read(count=q.size).reshape(seq, -1)
    assert np.isfinite(got[:seq - 2]).all()
    for t in range(seq):
        d1 = ctx.upload(q[t])
        ctx.attention(d1, kc, vc, total, one, 1, past + t, heads, kv_heads, kind="exact")
        np.testing.assert_array_equal(one.read(count=heads * 64), got[t], err_msg=f"query {t}")
        if t < seq - 2:
            np.testing.assert_array_equal(one.read(count=heads * 64).view(np.uint32), got[t].view(np.uint32))
        d1.free()
    for b in (kc, vc, dq, out, one):
        b.free()


@pytest.mark.parametrize("seq,past,heads,kv_heads", [
    (39, 0, 14, 2),       # 546 queries x heads, at most 512 + 39: a block each
    (40, 0, 14, 2),       # 560, more than 512 + 40: tiles
    (321, 0, 2, 1), (41, 471, 16, 2),                 # the second fills 512 positions
    (32, 481, 16, 2),     # past 512 positions 512 stay a block each,
    (33, 480, 16, 2), (48, 976, 14, 2),               # 528 go in tiles; 1024 filled
    (129, 896, 4, 4), (48, 2000, 14, 2),              # past 1024, and 2048 filled
    (44, 2010, 14, 2),    # past 2048: a block each again
])
def test_query_tiles_at_their_limits_equal_single_queries_bitwise(ctx, hip, seq, past, heads, kv_heads):
    test_query_tiles_equal_single_queries_bitwise(ctx, hip, seq, past, heads, kv_heads)


def test_query_tiles_keep_subnormal_products(ctx, hip):
    """One key holds nearly all of each query's probability and its value is 0; the other keys'
    probabilities are f32 subnormals (exp(-92) = 1.1e-40), and so is the whole output."""
    seq, heads = 48, 14
    k = np.full((2, seq, 64), -1.0, np.float16)
    k[:, 0] = 0.0
    v = np.zeros((2, 64, 64), np.float16)
    v[:, :, 1:seq] = np.random.default_rng(9).uniform(0.5, 2, (2, 64, seq - 1))
    q = np.full((seq, heads * 64), 11.5, np.float32)      # 64 * 11.5 / 8 = 92
    kc, vc, dq = ctx.upload(k), ctx.upload(v), ctx.upload(q)
    out, one = ctx.empty(q.nbytes), ctx.empty(heads * 64 * 4)
    ctx.attention(dq, kc, vc, seq, out, seq, 0, heads, 2, kind="exact")
    got = out.read(count=q.size).reshape(seq, -1)
    p = np.float32(np.exp(-92.0) / (1 + 47 * np.exp(-92.0)))
    assert 0 < p < np.finfo(np.float32).tiny and (got[1:] > 0).all()
    want = np.concatenate([v[h // 7, :, 1] for h in range(heads)]).astype(np.float32) * p
    np.testing.assert_allclose(got[1], want, rtol=0, atol=3e-45)      # p and the product: steps of 1.4e-45
    for t in range(seq):
        ctx.attention(dq, kc, vc, seq, one, 1, t, heads, 2, kind="exact")
        np.testing.assert_array_equal(one.read(count=heads * 64).view(np.uint32), got[t].view(np.uint32), err_msg=f"query {t}")
    for b in (kc, vc, dq, out, one):
        b.free()


@pytest.mark.parametrize("seq,heads,kv_heads", [(16, 14, 2), (64, 2, 1)])
def test_few_queries_after_a_long_past_cost_what_one_costs(ctx, hip, seq, heads, kv_heads):
    """Their (query, head) blocks are fewer than the CUs, so they take one query's time; a tile
    takes three times as long."""
    total = 1980 + seq
    rng = np.random.default_rng(4)
    kc = ctx.upload(rng.standard_normal((kv_heads, total, 64)).astype(np.float16))
    vc = ctx.upload(rng.standard_normal((kv_heads, 64, (total + 63) // 64 * 64)).astype(np.float16))
    dq, out = ctx.upload(rng.standard_normal((seq, heads * 64)).astype(np.float32)), ctx.empty(seq * heads * 64 * 4)

    def best(n, past):
        a, b, least = ctx.event(), ctx.event(), 1e9
        for _ in range(8):
            ctx.record(a)
            for _ in range(20):
                ctx.attention(dq, kc, vc, total, out, n, past, heads, kv_heads, kind="exact")
            ctx.record(b)
            least = min(least, ctx.elapsed_ms(a, b))
        ctx.destroy_event(a)
        ctx.destroy_event(b)
        return least
    assert best(seq, 1980) < 2 * best(1, total - 1)
    for b in (kc, vc, dq, out):
        b.free()
