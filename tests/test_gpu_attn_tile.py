"""Exact attention of a prompt by tiles of 16 queries (csrc/attention.h k_attn_tile): every query
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
