"""The batched prefill's contractions on the f32 matrix cores (csrc/chain.hip) against the decode
step: the same sums in the same order, so a prompt's logits and its f16 K/V rows are those of the
same positions stepped one at a time, bit for bit -- at the edges of the 64-position and 64-row
tiles, with one and several splits of the team's slots, ragged last chunks and every format."""
import ctypes
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", ["f16", "int8", "int4"])
@pytest.mark.parametrize("hidden,ffn,heads,kv_heads", [
    (128, 256, 2, 1),       # fewer chunks than lanes: empty slots in the tree
    (896, 4864, 14, 2),     # the 0.5B layer: 64-lane teams, several chunks per lane (down)
    (192, 1184, 3, 1),      # rows and chunks off the tiles
])
def test_batched_prefill_on_matrix_cores_equals_steps_bitwise(ctx, hip, scheme, hidden, ffn, heads, kv_heads):
    group = 32 if hidden == 192 else 128
    cfg = hip.ModelConfig(hidden=hidden, intermediate=ffn, layers=2, heads=heads, kv_heads=kv_heads, vocab=1000)
    ckpt = hip.synthesize_checkpoint(cfg, seed=21)
    model = hip.GpuModel.load(ctx, hip.device_tensors(ckpt, cfg, scheme, group, "int8"), cfg, maxPositions=512)
    ids = hip.synth_tokens(21, "chain", cfg.vocab, 300)
    steps = model.newCache(300)
    model.set_matmul("matvec")
    want = {}
    for t in range(300):
        if t + 1 in (12, 15, 24, 33, 64, 65, 129, 300):
            want[t + 1] = model.forward_tokens(ids[t:t + 1], steps)["logits"]
        else:
            model.forward_tokens(ids[t:t + 1], steps, wantLogits=False)
    kv = [steps.present(L) for L in range(cfg.layers)]
    model.set_matmul("batched")
    for n, logits in want.items():
        cache = model.newCache(300)
        got = model.forward_tokens(ids[:n], cache)["logits"]
        np.testing.assert_array_equal(got.view(np.uint32), logits.view(np.uint32), err_msg=f"{n} positions")
        for L in range(cfg.layers):
            p = cache.present(L)
            for name in ("key", "value"):
                np.testing.assert_array_equal(p[name], kv[L][name][:, :n], err_msg=f"{n} positions, layer {L} {name}")
        cache.destroy()
    # after a past of odd length
    cache = model.newCache(300)
    model.forward_tokens(ids[:35], cache, wantLogits=False)
    got = model.forward_tokens(ids[35:129], cache)["logits"]
    np.testing.assert_array_equal(got.view(np.uint32), want[129].view(np.uint32))
    cache.destroy()
    steps.destroy()
    model.destroy()


@pytest.mark.parametrize("scheme", ["f16", "int8", "int4"])
@pytest.mark.parametrize("hidden,ffn,heads", [
    (1024, 8192, 16),       # the widest fast model: the deepest tree with several chunks a lane
    (512, 1536, 8),         # int4 down: a team of 64 lanes cut once; gate|up: one of 32, whole
])
def test_batched_prefill_deepest_trees_equal_steps_bitwise(ctx, hip, scheme, hidden, ffn, heads):
    cfg = hip.ModelConfig(hidden=hidden, intermediate=ffn, layers=2, heads=heads, kv_heads=2, vocab=1000)
    model = hip.GpuModel.load(ctx, hip.device_tensors(hip.synthesize_checkpoint(cfg, seed=27), cfg, scheme, 128, "int8"),
                              cfg, maxPositions=512)
    ids = hip.synth_tokens(27, "chain.deep", cfg.vocab, 512)
    steps = model.newCache(512)
    model.set_matmul("matvec")
    want = {n: model.forward_tokens(ids[a:n], steps)["logits"] for a, n in ((0, 65), (65, 319), (319, 512))}
    model.set_matmul("batched")
    for n, logits in want.items():
        cache = model.newCache(512)
        got = model.forward_tokens(ids[:n], cache)["logits"]
        np.testing.assert_array_equal(got.view(np.uint32), logits.view(np.uint32), err_msg=f"{n} positions")
        for L in range(cfg.layers):
            p, s = cache.present(L), steps.present(L)
            for name in ("key", "value"):
                np.testing.assert_array_equal(p[name], s[name][:, :n], err_msg=f"{n} positions, layer {L} {name}")
        cache.destroy()
    steps.destroy()
    model.destroy()


@pytest.mark.parametrize("fmt", ["f16", "int8", "int4"])
@pytest.mark.parametrize("rows,cols,group", [
    (1, 128, 128),          # one row: a tile of clamped rows
    (17, 896, 128),         # one row past a tile; 56 / 28 / 112 chunks
    (128, 4864, 128),       # several chunks per lane, a ragged last pass
    (70, 1184, 32),         # chunks off the slabs
])
def test_exact_matvec_on_matrix_cores_equals_single_positions_bitwise(ctx, hip, fmt, rows, cols, group):
    """qh_matvec from 6 positions runs on the f64 matrix cores: each position's outputs are those
    of the one-position call, bit for bit (int4 zero points off the quantizer's integers too)."""
    rng = np.random.default_rng(rows + cols)
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    if fmt == "f16":
        bufs = [ctx.upload(w.astype(np.float16).view(np.uint16))]
        W = ctx.weight(hip.FMT_F16, rows, cols, bufs[0])
    elif fmt == "int8":
        q, s = hip.quantize_int8(w)
        q[0, :3] = -128
        bufs = [ctx.upload(q), ctx.upload(s)]
        W = ctx.weight(hip.FMT_INT8, rows, cols, *bufs)
    else:
        q, s, z = hip.quantize_int4(w, group)
        z[0, 0] = 3.5
        bufs = [ctx.upload(q), ctx.upload(s), ctx.upload(z)]
        W = ctx.weight(hip.FMT_INT4, rows, cols, *bufs, group)
    bias = ctx.upload(rng.standard_normal(rows).astype(np.float32))
    x = rng.standard_normal((49, cols)).astype(np.float32)
    dy = ctx.empty(49 * rows * 4)
    want = np.empty((49, rows), np.float32)
    for t in range(49):
        dx = ctx.upload(x[t])
        ctx.matvec(W, dx, bias, dy, 1)
        want[t] = dy.read(count=rows)
        dx.free()
    dx = ctx.upload(x)
    for seq in (6, 8, 16, 17, 32, 33, 49):
        ctx.matvec(W, dx, bias, dy, seq)
        np.testing.assert_array_equal(dy.read(count=seq * rows).view(np.uint32), want[:seq].reshape(-1).view(np.uint32),
                                      err_msg=f"{seq} positions")
    for b in bufs + [bias, dx, dy]:
        b.free()


@pytest.mark.parametrize("fmt", ["f16", "int8", "int4"])
@pytest.mark.parametrize("rows,cols,seqs", [
    (1361, 256, (16, 32, 33, 48)),     # 86 row blocks: 32 positions a tile of 16 per block, 33 two
    (4097, 1184, (6, 17, 31)),         # 257: two tiles per block from 17 positions
])
def test_exact_matvec_tiles_per_block_equal_single_positions_bitwise(ctx, hip, fmt, rows, cols, seqs):
    """A block takes one or two tiles of 16 positions, by how many blocks there are."""
    rng = np.random.default_rng(rows)
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    if fmt == "f16":
        bufs = [ctx.upload(w.astype(np.float16).view(np.uint16))]
        W = ctx.weight(hip.FMT_F16, rows, cols, bufs[0])
    elif fmt == "int8":
        bufs = [ctx.upload(a) for a in hip.quantize_int8(w)]
        W = ctx.weight(hip.FMT_INT8, rows, cols, *bufs)
    else:
        bufs = [ctx.upload(a) for a in hip.quantize_int4(w, 32)]
        W = ctx.weight(hip.FMT_INT4, rows, cols, *bufs, 32)
    n = max(seqs)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    dy = ctx.empty(n * rows * 4)
    want = np.empty((n, rows), np.float32)
    for t in range(n):
        dx = ctx.upload(x[t])
        ctx.matvec(W, dx, None, dy, 1)
        want[t] = dy.read(count=rows)
        dx.free()
    dx = ctx.upload(x)
    for seq in seqs:
        ctx.matvec(W, dx, None, dy, seq)
        np.testing.assert_array_equal(dy.read(count=seq * rows).view(np.uint32), want[:seq].reshape(-1).view(np.uint32),
                                      err_msg=f"{seq} positions")
    for b in bufs + [dx, dy]:
        b.free()


def test_prompt_attention_past_1024_positions_equals_steps_bitwise(ctx, hip):
    """Slots of several chunks (four states a slot), and the step from one chunk a slot to two, in
    the prompt's merged attention: the decode steps' logits and K/V rows bit for bit."""
    cfg = hip.ModelConfig(hidden=256, intermediate=256, layers=2, heads=4, kv_heads=2, vocab=1000)
    model = hip.GpuModel.load(ctx, hip.device_tensors(hip.synthesize_checkpoint(cfg, seed=22), cfg, "int8", 128, "int8"),
                              cfg, maxPositions=2300)
    ids = hip.synth_tokens(22, "chain.long", cfg.vocab, 2250)
    steps, cache = model.newCache(2300), model.newCache(2300)
    model.set_matmul("matvec")
    want = {}
    for a, b in ((0, 1010), (1010, 1040), (1040, 2040), (2040, 2250)):
        want[b] = model.forward_tokens(ids[a:b], steps)["logits"]
    model.set_matmul("batched")
    for a, b in ((0, 1010), (1010, 1040), (1040, 2040), (2040, 2250)):
        got = model.forward_tokens(ids[a:b], cache)["logits"]
        np.testing.assert_array_equal(got.view(np.uint32), want[b].view(np.uint32), err_msg=f"to {b}")
    for L in range(cfg.layers):
        p, s = cache.present(L), steps.present(L)
        np.testing.assert_array_equal(p["key"], s["key"])
        np.testing.assert_array_equal(p["value"], s["value"])
    cache.destroy()
    steps.destroy()
    model.destroy()


def test_short_prompts_after_a_past_equal_steps_bitwise(ctx, hip):
    """Few queries over a long context take the decode step's blocks and a merge, others a block per
    query and kv head: the steps' logits and K/V rows in both, on both sides of the line."""
    cfg = hip.ModelConfig(hidden=256, intermediate=256, layers=2, heads=4, kv_heads=2, vocab=1000)
    model = hip.GpuModel.load(ctx, hip.device_tensors(hip.synthesize_checkpoint(cfg, seed=25), cfg, "int8", 128, "int8"),
                              cfg, maxPositions=2300)
    ids = hip.synth_tokens(25, "chain.after", cfg.vocab, 2300)
    steps, cache = model.newCache(2300), model.newCache(2300)
    done = 0
    for n in (100, 2, 190, 2, 9, 800, 40, 64, 128, 700, 40, 64, 129, 2, 9):
        model.set_matmul("matvec")
        want = model.forward_tokens(ids[done:done + n], steps)["logits"]
        model.set_matmul("batched")
        got = model.forward_tokens(ids[done:done + n], cache)["logits"]
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32), err_msg=f"{n} after {done}")
        done += n
    for L in range(cfg.layers):
        p, s = cache.present(L), steps.present(L)
        np.testing.assert_array_equal(p["key"], s["key"])
        np.testing.assert_array_equal(p["value"], s["value"])
    cache.destroy()
    steps.destroy()
    model.destroy()


def test_short_prompts_after_a_long_past_cost_what_they_cost_at_first(ctx, hip):
    """Two queries over 8000 positions: 16 blocks each share the context, where one block each would
    more than double the forward."""
    cfg = hip.ModelConfig(hidden=256, intermediate=256, layers=8, heads=4, kv_heads=1, vocab=1000)
    model = hip.GpuModel.load(ctx, hip.device_tensors(hip.synthesize_checkpoint(cfg, seed=26), cfg, "int8", 128, "int8"),
                              cfg, maxPositions=8192)
    ids = hip.synth_tokens(26, "chain.long.past", cfg.vocab, 8000)
    cache = model.newCache(8192)
    model.forward_tokens(ids, cache, wantLogits=False)

    def best(past):
        least = 1e9
        for _ in range(30):
            cache.length = past
            start = time.perf_counter()
            model.forward_tokens(ids[:2], cache)
            least = min(least, time.perf_counter() - start)
        return least
    late = best(8000)
    assert late < 1.6 * best(0)
    cache.destroy()
    model.destroy()


@pytest.mark.parametrize("fmt", ["f16", "int8", "int4"])
@pytest.mark.parametrize("cols", [896, 4864])     # positions in LDS; an f64 copy of all of them
def test_matvec_of_unaligned_positions_equals_single_positions_bitwise(ctx, hip, fmt, cols):
    """x off its 16 bytes stays in tiles of 8, 4, 2 and 1 positions."""
    rng = np.random.default_rng(cols)
    w = (rng.standard_normal((21, cols)) * 0.02).astype(np.float32)
    if fmt == "f16":
        bufs = [ctx.upload(w.astype(np.float16).view(np.uint16))]
        W = ctx.weight(hip.FMT_F16, 21, cols, bufs[0])
    elif fmt == "int8":
        bufs = [ctx.upload(a) for a in hip.quantize_int8(w)]
        W = ctx.weight(hip.FMT_INT8, 21, cols, *bufs)
    else:
        bufs = [ctx.upload(a) for a in hip.quantize_int4(w, 128)]
        W = ctx.weight(hip.FMT_INT4, 21, cols, *bufs, 128)
    x = rng.standard_normal((19, cols)).astype(np.float32)
    dx = ctx.upload(np.concatenate([[np.float32(0)], x.reshape(-1)]))
    off = hip.DeviceBuffer(ctx, dx.ptr + 4, dx.nbytes - 4)
    dy = ctx.empty(19 * 21 * 4)
    want = np.empty((19, 21), np.float32)
    for t in range(19):
        one = ctx.upload(x[t])
        ctx.matvec(W, one, None, dy, 1)
        want[t] = dy.read(count=21)
        one.free()
    for seq in (1, 6, 7, 8, 11, 16, 19):
        ctx.matvec(W, off, None, dy, seq)
        np.testing.assert_array_equal(dy.read(count=seq * 21).view(np.uint32), want[:seq].reshape(-1).view(np.uint32),
                                      err_msg=f"{seq} positions")
    for b in bufs + [dx, dy]:
        b.free()


def test_exact_workspace_holds_no_f64_copy_of_a_prompt(ctx, hip):
    """512 positions of 4864 ffn columns would be 20 MB that no launch reads: from 6 positions the
    exact contractions read the f32 rows."""
    rt = ctypes.CDLL("libamdhip64.so")
    rt.hipMemGetInfo.argtypes = [ctypes.POINTER(ctypes.c_size_t)] * 2

    def free_bytes():
        ctx.done()
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert rt.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value
    cfg = hip.ModelConfig(hidden=128, intermediate=4864, layers=1, heads=2, kv_heads=1, vocab=1000)
    model = hip.GpuModel.load(ctx, hip.device_tensors(hip.synthesize_checkpoint(cfg, seed=24), cfg, "int8", 128, "int8"),
                              cfg, maxPositions=512, numerics="exact")
    cache = model.newCache(512)
    ids = hip.synth_tokens(24, "chain.workspace", cfg.vocab, 5)
    before = free_bytes()
    model.forward_tokens(ids, cache)               # in tiles, which read the copy
    assert before - free_bytes() < 1.25 * 512 * 4 * (7 * 128 + 3 * 4864)
    cache.destroy()
    model.destroy()


def test_short_prompts_of_a_narrow_model_cost_what_eight_positions_cost(ctx, hip):
    """64 positions through 512-column int4 layers are one launch of tiles per contraction, as 8 are;
    on the matrix cores they would take twice as long."""
    cfg = hip.ModelConfig(hidden=512, intermediate=1536, layers=4, heads=8, kv_heads=2, vocab=1000)
    model = hip.GpuModel.load(ctx, hip.device_tensors(hip.synthesize_checkpoint(cfg, seed=23), cfg, "int4", 128, "int8"),
                              cfg, maxPositions=64)
    ids = hip.synth_tokens(23, "chain.narrow", cfg.vocab, 64)
    cache = model.newCache(64)

    def best(n):
        least = 1e9
        for _ in range(30):
            cache.length = 0
            start = time.perf_counter()
            model.forward_tokens(ids[:n], cache)
            least = min(least, time.perf_counter() - start)
        return least
    assert best(64) < 1.5 * best(8)
    cache.destroy()
    model.destroy()
