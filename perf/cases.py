"""The work that is timed when this library is made faster: calls a program makes through its
public entry points, from one position's elementwise operators to a whole prompt, with the
inputs, an f64 evaluation of each in plain torch, and the bytes and operations each cannot do
without. The sizes are those of the Qwen2.5-0.5B shape this engine runs (and, drawn, generic
and ragged ones around it)."""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llm-inference-webgpu_amd"))
import qwen_hip as H  # noqa: E402

CFG = H.QWEN25_05B
HIDDEN, FFN, VOCAB, HD = CFG.hidden, CFG.intermediate, CFG.vocab, CFG.head_dim
LAYER_SHAPES = ((896, 896), (128, 896), (4864, 896), (896, 4864))
FMT = {"f16": H.FMT_F16, "int8": H.FMT_INT8, "int4": H.FMT_INT4}
GROUP = 128


def listed():
    return [
        # One position's elementwise operators, as the reference's model loop issues them between
        # the matvecs: the smallest calls, bound by launches.
        {"name": "glue-1", "kind": "glue", "rows": 1},
        # MATVEC / batchedMatvec on its own: the reference's 52-token prompt through the gate
        # projection, and the loop's exact (f64) sums.
        {"name": "matvec-int8-4864x896-52", "kind": "matvec", "fmt": "int8", "rows": 4864, "cols": 896, "seq": 52},
        # The isolated weight-only int8 matvec, one launch over the 24 layers' gate and up matrices.
        {"name": "matvec-list-48", "kind": "list", "rows": 4864, "cols": 896, "count": 48},
        # The prompt contraction on the matrix cores, one gate projection of a 512-token prompt.
        {"name": "matmul-int8-4864x896-512", "kind": "matmul", "fmt": "int8", "rows": 4864, "cols": 896, "seq": 512},
        # Decode attention of one query over long caches (streams being served side by side).
        {"name": "attn-list-4096x64", "kind": "attn", "how": "list", "ctx": 4096, "count": 64, "heads": 14, "kv": 2},
        # A 512-token prompt's attention, in the CPU path's order and on the matrix cores.
        {"name": "attn-exact-512", "kind": "attn", "how": "exact", "past": 0, "seq": 512, "heads": 14, "kv": 2},
        {"name": "attn-mfma-1024", "kind": "attn", "how": "mfma", "past": 0, "seq": 1024, "heads": 14, "kv": 2},
        # Loading: all layers' gate and up projections, bf16 as stored, to int4.
        {"name": "quantize-int4-gate-up", "kind": "quantize", "src": "bf16", "to": "int4", "rows": 233472, "cols": 896},
        # A prompt to its first token, in the default mode and on the matrix cores.
        {"name": "prefill-batched-int8-512", "kind": "prefill", "scheme": "int8", "matmul": "batched", "seq": 512},
        {"name": "prefill-mfma-int8-512", "kind": "prefill", "scheme": "int8", "matmul": "mfma", "seq": 512},
        # Greedy decoding, the headline configuration: int4 layers, int8 head, context 1024.
        {"name": "decode-int4-1024", "kind": "decode", "scheme": "int4", "ctx": 1024, "steps": 16},
        # Perplexity of a passage, one position's logits after another.
        {"name": "score-int4-128", "kind": "score", "scheme": "int4", "seq": 128},
    ]


def _logint(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("glue", "matvec", "matvec", "list", "matmul", "matmul", "attn", "attn", "attn", "quantize",
                       "prefill", "prefill", "decode", "score"))
    shape = rng.choice(LAYER_SHAPES + ((_logint(rng, 16, 5000), 128 * rng.randint(1, 38)),))
    heads, kv = rng.choice(((14, 2), (14, 2), (8, 2), (4, 4)))
    if kind == "glue":
        return {"kind": kind, "rows": _logint(rng, 1, 512)}
    if kind == "matvec":
        return {"kind": kind, "fmt": rng.choice(("f16", "int8", "int4")), "rows": shape[0], "cols": shape[1],
                "seq": _logint(rng, 1, 256)}
    if kind == "list":
        return {"kind": kind, "rows": shape[0], "cols": shape[1],
                "count": _logint(rng, 1, max(1, min(512, (256 << 20) // (shape[0] * shape[1]))))}
    if kind == "matmul":
        return {"kind": kind, "fmt": rng.choice(("int8", "int4")), "rows": shape[0], "cols": shape[1],
                "seq": _logint(rng, 8, 512)}
    if kind == "attn":
        how = rng.choice(("list", "splitk", "exact", "mfma"))
        if how == "list":
            ctx = _logint(rng, 64, 32768)
            return {"kind": kind, "how": how, "ctx": ctx, "count": _logint(rng, 1, max(1, min(512, 262144 // ctx))),
                    "heads": heads, "kv": kv}
        if how == "splitk":
            return {"kind": kind, "how": how, "past": _logint(rng, 16, 32000), "seq": rng.choice((1, 1, 2, 5, 8)),
                    "heads": heads, "kv": kv}
        return {"kind": kind, "how": how, "past": rng.choice((0, 0, _logint(rng, 16, 1024))),
                "seq": _logint(rng, 1, 512 if how == "exact" else 1024), "heads": heads, "kv": kv}
    if kind == "quantize":
        return {"kind": kind, "src": rng.choice(("bf16", "bf16", "f32")), "to": rng.choice(("f16", "int8", "int4")),
                "rows": _logint(rng, 16, 65536), "cols": rng.choice((896, 4864, 128 * rng.randint(1, 38)))}
    scheme = rng.choice(("int8", "int4", "f16"))
    if kind == "prefill":
        return {"kind": kind, "scheme": scheme, "matmul": rng.choice(("batched", "mfma")), "seq": _logint(rng, 2, 512)}
    if kind == "decode":
        return {"kind": kind, "scheme": scheme, "ctx": _logint(rng, 16, 2048), "steps": rng.randint(3, 20)}
    return {"kind": kind, "scheme": scheme, "seq": _logint(rng, 8, 128)}


# ------------------------------------------------------------------ inputs --

_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        torch.cuda.init()
        _ctx = H.GpuContext.create(torch.cuda.current_device())
    return _ctx


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFFFFFF)


def _randn(g, *shape, std=1.0, dtype=torch.float32):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).to(dtype)


def _buf(t):
    return H.DeviceBuffer(_context(), t.data_ptr(), t.numel() * t.element_size())


def _rha(t):
    """Round half away from zero."""
    return torch.trunc(t + torch.copysign(torch.full_like(t, 0.5), t))


def _const(v):
    """A divisor on the GPU (torch multiplies by the reciprocal of a plain number)."""
    return torch.tensor([float(v)], dtype=torch.float64, device="cuda")


def _quantize(w, scheme):
    """The reference quantizer on f32 values [rows, cols]: (codes or packed bytes, scales, zeros),
    codes from the f64 scale, the scales stored f32."""
    rows, cols = w.shape
    if scheme == "f16":
        return w.to(torch.float16), None, None
    if scheme == "int8":
        scale = w.abs().amax(1).double() / _const(127)
        inv = torch.where(scale > 0, _const(1) / scale, torch.zeros_like(scale))
        q = _rha(w.double() * inv[:, None]).clamp_(-127, 127).to(torch.int8)
        return q, scale.float(), None
    g = w.double().reshape(rows, cols // GROUP, GROUP)
    lo, hi = g.amin(2).clamp(max=0), g.amax(2).clamp(min=0)
    scale = (hi - lo) / _const(15)
    inv = torch.where(scale > 0, _const(1) / scale, torch.zeros_like(scale))
    zero = torch.where(scale > 0, _rha(-lo / scale), torch.zeros_like(scale)).clamp_(0, 15)
    q = (_rha(g * inv[:, :, None]) + zero[:, :, None]).clamp_(0, 15).to(torch.uint8).reshape(rows, cols // 2, 2)
    return q[:, :, 0] | (q[:, :, 1] << 4), scale.float(), zero.float()


def _dequantize(q, s, z, scheme):
    """The f64 weights the stored codes stand for."""
    if scheme == "f16":
        return q.double()
    if scheme == "int8":
        return q.double() * s.double()[:, None]
    rows = q.shape[0]
    lv = torch.stack((q & 15, q >> 4), 2).reshape(rows, -1, GROUP).double()
    return ((lv - z.double()[:, :, None]) * s.double()[:, :, None]).reshape(rows, -1)


def _rope_tables(positions):
    inv = CFG.rope_theta ** (-torch.arange(0, HD, 2, dtype=torch.float64, device="cuda") / HD)
    a = torch.arange(positions, dtype=torch.float64, device="cuda")[:, None] * inv[None]
    return a.cos(), a.sin()


def _inputs(case, seed):
    """The tensors of an operator's call."""
    g, k = _gen(seed), case["kind"]
    if k == "glue":
        n = case["rows"]
        return {"x": _randn(g, n, HIDDEN), "gain": 1 + _randn(g, HIDDEN, std=0.1), "q": _randn(g, n, HIDDEN),
                "k": _randn(g, n, CFG.kv_dim), "v": _randn(g, n, CFG.kv_dim), "gate": _randn(g, n, FFN),
                "up": _randn(g, n, FFN), "delta": _randn(g, n, HIDDEN)}
    if k in ("matvec", "matmul"):
        q, s, z = _quantize(_randn(g, case["rows"], case["cols"], std=0.02), case["fmt"])
        return {"q": q, "s": s, "z": z, "x": _randn(g, case["seq"], case["cols"]), "b": _randn(g, case["rows"], std=0.02)}
    if k == "list":
        n, r, c = case["count"], case["rows"], case["cols"]
        q = torch.empty((n, r, c), dtype=torch.int8, device="cuda")
        s = torch.empty((n, r), dtype=torch.float32, device="cuda")
        for i in range(n):
            q[i], s[i], _ = _quantize(_randn(g, r, c, std=0.02), "int8")
        return {"q": q, "s": s, "x": _randn(g, n, c, dtype=torch.float16)}
    if k == "attn":
        n, total = case.get("count", 1), _total(case)
        seq = case.get("seq", 1)
        vs = (total + 63) // 64 * 64
        v = torch.zeros((n, case["kv"], HD, vs), dtype=torch.float16, device="cuda")
        v[..., :total] = _randn(g, n, case["kv"], HD, total, dtype=torch.float16)
        return {"q": _randn(g, seq, case["heads"] * HD), "k": _randn(g, n, case["kv"], total, HD, dtype=torch.float16), "v": v}
    w = _randn(g, case["rows"], case["cols"], std=0.02)
    return {"w": w.to(torch.bfloat16) if case["src"] == "bf16" else w}


def _total(case):
    return case["ctx"] if case["how"] == "list" else case["past"] + case["seq"]


def _checkpoint(seed):
    """bf16 tensors of the architecture, on the GPU: N(0, 0.02), norm gains 1."""
    g = _gen(seed)
    out = {}
    for name, shape in CFG.expected_tensors().items():
        if name.endswith("norm.weight"):
            out[name] = torch.ones(shape, dtype=torch.bfloat16, device="cuda")
        else:
            out[name] = _randn(g, *shape, std=0.02, dtype=torch.bfloat16)
    return out


def _head_scheme(scheme):
    return "f16" if scheme == "f16" else "int8"


def _ids(seed, n):
    return np.random.RandomState((int(seed) * 2654435761 + 12345) % (1 << 32)).randint(0, VOCAB, n).astype(np.int32)


class _Model:
    """A loaded model with a cache, freed with the state that holds it."""

    def __init__(self, case, seed):
        ckpt = {n: t.view(torch.int16).cpu().numpy().view(np.uint16) if t.ndim > 1 else t.float().cpu().numpy()
                for n, t in _checkpoint(seed).items()}
        total = case["ctx"] + case["steps"] + 1 if case["kind"] == "decode" else case["seq"]
        self.model = H.GpuModel.load_checkpoint(_context(), ckpt, CFG, scheme=case["scheme"], group=GROUP,
                                                lm_head=_head_scheme(case["scheme"]), maxPositions=max(64, total),
                                                matmul=case.get("matmul", "batched"))
        self.cache = self.model.newCache(max(64, total))

    def __del__(self):
        if getattr(self, "cache", None) is not None:
            self.cache.destroy()
        if getattr(self, "model", None) is not None:
            self.model.destroy()


def prepare(case, seed):
    ctx, k = _context(), case["kind"]
    if k in ("prefill", "score"):
        return {"case": case, "m": _Model(case, seed), "ids": _ids(seed, case["seq"])}
    if k == "decode":
        m = _Model(case, seed)
        first = m.model.forward_tokens(_ids(seed, case["ctx"]), m.cache)["argmax"]
        m.model.decode_prepare(m.cache)
        return {"case": case, "m": m, "first": first}
    s = {"case": case, "t": _inputs(case, seed)}
    t = s["t"]
    b = s["b"] = {n: _buf(x) for n, x in t.items() if x is not None}
    e = lambda *shape, dtype=torch.float32: torch.zeros(shape, dtype=dtype, device="cuda")  # noqa: E731
    if k == "glue":
        n = case["rows"]
        cos, sin = _rope_tables(2 * n)
        t["cos"], t["sin"] = cos.float(), sin.float()
        o = {"norm": e(n, HIDDEN), "q": e(n, HIDDEN), "gate": e(n, FFN), "x": e(n, HIDDEN),
             "keys": e(CFG.kv_heads, 2 * n, HD, dtype=torch.float16),
             "values": e(CFG.kv_heads, HD, (2 * n + 63) // 64 * 64, dtype=torch.float16)}
        b["cos"], b["sin"] = _buf(t["cos"]), _buf(t["sin"])
    elif k in ("matvec", "matmul"):
        o = {"y": e(case["seq"], case["rows"])}
        s["w"] = ctx.weight(FMT[case["fmt"]], case["rows"], case["cols"], b["q"], b.get("s"), b.get("z"),
                            GROUP if case["fmt"] == "int4" else 0)
    elif k == "list":
        o = {"y": e(case["count"], case["rows"])}
        s["w"] = ctx.weight(H.FMT_INT8, case["rows"], case["cols"], b["q"], b["s"])
    elif k == "attn":
        o = {"out": e(case.get("count", case.get("seq", 1)), case["heads"] * HD)}
    else:
        rows, cols, to = case["rows"], case["cols"], case["to"]
        o = {"data": e(rows, cols, dtype=torch.float16) if to == "f16" else
             e(rows, cols, dtype=torch.int8) if to == "int8" else e(rows, cols // 2, dtype=torch.uint8)}
        if to == "int8":
            o["scales"] = e(rows)
        if to == "int4":
            o["scales"], o["zeros"] = e(rows, cols // GROUP), e(rows, cols // GROUP)
    s["out"] = o
    s["o"] = {n: _buf(x) for n, x in o.items()}
    return s


def run(s):
    ctx, case = _context(), s["case"]
    k = case["kind"]
    if k == "prefill":
        m = s["m"]
        m.cache.length = 0
        r = m.model.forward_tokens(s["ids"], m.cache)
        return {"logits": r["logits"], "argmax": r["argmax"], "present": m.cache.present(CFG.layers - 1)}
    if k == "score":
        m = s["m"]
        m.cache.length = 0
        return {"nll": m.model.score(s["ids"], m.cache), "present": m.cache.present(CFG.layers - 1)}
    if k == "decode":
        m = s["m"]
        m.cache.length = case["ctx"]
        tokens = m.model.decode(m.cache, s["first"], case["steps"])
        return {"tokens": tokens, "logits": m.cache.vector("logits")}
    b, o = s["b"], s["o"]
    if k == "glue":
        n = case["rows"]
        ctx.rmsnorm(b["x"], b["gain"], o["norm"], n, HIDDEN, CFG.eps)
        ctx.copy(b["q"], 0, o["q"], 0, b["q"].nbytes)
        ctx.rope(o["q"], b["cos"], b["sin"], 2 * n, n, CFG.heads, HD, n)
        ctx.kv_append(b["k"], b["v"], o["keys"], o["values"], 2 * n, CFG.kv_heads, HD, n, n)
        ctx.copy(b["gate"], 0, o["gate"], 0, b["gate"].nbytes)
        ctx.swiglu(o["gate"], b["up"], n * FFN)
        ctx.copy(b["x"], 0, o["x"], 0, b["x"].nbytes)
        ctx.add(o["x"], b["delta"], n * HIDDEN)
    elif k == "matvec":
        ctx.matvec(s["w"], b["x"], b["b"], o["y"], case["seq"])
    elif k == "matmul":
        ctx.matmul_prefill(s["w"], b["x"], b["b"], o["y"], case["seq"])
    elif k == "list":
        r, c = case["rows"], case["cols"]
        ctx.matvec_xh_list(s["w"], case["count"], r * c, r, b["x"], c, o["y"])
    elif k == "attn":
        total, h, kv = _total(case), case["heads"], case["kv"]
        if case["how"] == "list":
            vs = s["t"]["v"].shape[-1]
            ctx.attention_list(b["q"], b["k"], b["v"], kv * total * HD, kv * HD * vs, case["count"], total, o["out"],
                               total - 1, h, kv)
        else:
            ctx.attention(b["q"], b["k"], b["v"], total, o["out"], case["seq"], case["past"], h, kv, kind=case["how"])
    else:
        ctx.quantize(b["w"], H.FMT_BF16 if case["src"] == "bf16" else H.FMT_F32, case["rows"], case["cols"],
                     FMT[case["to"]], GROUP if case["to"] == "int4" else 0, o["data"], o.get("scales"), o.get("zeros"))
    return s["out"]


# ------------------------------------------------------ bytes and operations --

def _wbytes(rows, cols, fmt):
    return rows * cols * 2 if fmt == "f16" else rows * (cols + 4) if fmt == "int8" else rows * (cols // 2 + 8 * (cols // GROUP))


def _layer_params():
    return 2 * HIDDEN * HIDDEN + 2 * CFG.kv_dim * HIDDEN + 3 * FFN * HIDDEN


def _model_bytes(scheme):
    per = sum(_wbytes(r, c, scheme) for r, c in ((HIDDEN, HIDDEN),) * 2 + ((CFG.kv_dim, HIDDEN),) * 2
              + ((FFN, HIDDEN),) * 2 + ((HIDDEN, FFN),))
    return CFG.layers * per + _wbytes(VOCAB, HIDDEN, _head_scheme(scheme))


def work(case):
    k = case["kind"]
    if k == "glue":
        n = case["rows"]
        return {"bytes": n * (4 * (7 * HIDDEN + 2 * CFG.kv_dim + 3 * FFN + HD) + 4 * CFG.kv_dim), "flops": n * (12 * HIDDEN + 6 * FFN)}
    if k in ("matvec", "matmul"):
        r, c, n = case["rows"], case["cols"], case["seq"]
        return {"bytes": _wbytes(r, c, case["fmt"]) + 4 * n * (r + c) + 4 * r, "flops": 2 * n * r * c}
    if k == "list":
        r, c, n = case["rows"], case["cols"], case["count"]
        return {"bytes": n * (r * c + 8 * r + 2 * c), "flops": 2 * n * r * c}
    if k == "attn":
        n, seq, total = case.get("count", 1), case.get("seq", 1), _total(case)
        keys = seq * (total - seq) + seq * (seq + 1) // 2
        return {"bytes": n * 4 * case["kv"] * HD * total + 8 * n * seq * case["heads"] * HD,
                "flops": 4 * n * keys * case["heads"] * HD}
    if k == "quantize":
        r, c = case["rows"], case["cols"]
        return {"bytes": r * c * (2 if case["src"] == "bf16" else 4) + _wbytes(r, c, case["to"]), "flops": 3 * r * c}
    kv = CFG.layers * 4 * CFG.kv_dim
    if k == "decode":
        n, ctx = case["steps"], case["ctx"]
        keys = n * ctx + n * (n + 1) // 2
        return {"bytes": n * _model_bytes(case["scheme"]) + kv * keys,
                "flops": 2 * n * (CFG.layers * _layer_params() + VOCAB * HIDDEN) + 4 * keys * HIDDEN * CFG.layers}
    n = case["seq"] if k == "prefill" else case["seq"] - 1
    heads = 1 if k == "prefill" else n
    return {"bytes": _model_bytes(case["scheme"]) + kv * n,
            "flops": 2 * (n * CFG.layers * _layer_params() + heads * VOCAB * HIDDEN) + 2 * n * (n + 1) * HIDDEN * CFG.layers}


# -------------------------------------------------------------- tolerances --

def tolerance(case):
    k = case["kind"]
    if k == "quantize":
        return "exact"
    if k == "glue":
        return {"rel": 1e-6}
    if k == "matvec":
        return {"rel": 1e-6}
    if k in ("matmul", "list"):  # 1.2e-7 and 7e-8 against f64
        return {"rel": 1e-6}
    if k == "attn":  # 2e-7 (exact order), 3e-7 (split-K, flash) against f64
        return {"rel": 1e-6} if case["how"] == "exact" else {"rel": 2e-6}
    # A whole model: an f16 cache entry that rounds the other way moves the layers after it
    # (logits up to 1.3e-4, the last layer's cache 3e-4 against f64).
    return {"rel": 1e-3, "differ": 0.0}


# ------------------------------------------------------------ f64 evaluation --

def _attend(q, keys, values, past):
    """Causal GQA attention in f64: q [seq, heads, 64], keys / values [kv, total, 64]."""
    seq, heads, _ = q.shape
    kv, total, _ = keys.shape
    out = torch.empty_like(q)
    mask = torch.arange(total, device="cuda")[None] > (past + torch.arange(seq, device="cuda"))[:, None]
    for h in range(heads):
        g = h // (heads // kv)
        p = (q[:, h] @ keys[g].T.contiguous()) / math.sqrt(HD)
        out[:, h] = torch.softmax(p.masked_fill(mask, -math.inf), 1) @ values[g]
    return out


class _Exact:
    """The model in f64 over the stored weights and an f16 cache."""

    def __init__(self, case, seed):
        scheme = case["scheme"]
        ck = _checkpoint(seed)
        self.w = {}
        for n, t in ck.items():
            w = t.float()
            self.w[n] = w.double() if w.ndim == 1 or "embed" in n else _dequantize(*_quantize(w, scheme), scheme)
        hs = _head_scheme(scheme)
        self.head = _dequantize(*_quantize(ck["model.embed_tokens.weight"].float(), hs), hs)
        self.kv = [None] * CFG.layers

    def forward(self, ids, rows=None):
        """Logits of the last position, or of every one; the cache grows."""
        w = self.w
        norm = lambda x, g: x / torch.sqrt((x * x).mean(1, keepdim=True) + CFG.eps) * g  # noqa: E731
        x = w["model.embed_tokens.weight"][torch.from_numpy(np.asarray(ids, np.int64)).cuda()]
        n = x.shape[0]
        past = 0 if self.kv[0] is None else self.kv[0][0].shape[1]
        cos, sin = (t[past:, None] for t in _rope_tables(past + n))
        rot = lambda t: torch.cat((t[..., :32] * cos - t[..., 32:] * sin, t[..., 32:] * cos + t[..., :32] * sin), 2)  # noqa: E731
        for i in range(CFG.layers):
            p = f"model.layers.{i}."
            a = norm(x, w[p + "input_layernorm.weight"])
            q, k, v = (a @ w[p + f"self_attn.{c}_proj.weight"].T + w[p + f"self_attn.{c}_proj.bias"] for c in "qkv")
            k = rot(k.reshape(n, CFG.kv_heads, HD)).half().double().transpose(0, 1).contiguous()
            v = v.reshape(n, CFG.kv_heads, HD).half().double().transpose(0, 1).contiguous()
            if past:
                k, v = (torch.cat(t, 1) for t in zip(self.kv[i], (k, v)))
            self.kv[i] = (k, v)
            o = _attend(rot(q.reshape(n, CFG.heads, HD)), k, v, past).reshape(n, HIDDEN)
            x = x + o @ w[p + "self_attn.o_proj.weight"].T
            a = norm(x, w[p + "post_attention_layernorm.weight"])
            gate, up = (a @ w[p + f"mlp.{c}_proj.weight"].T for c in ("gate", "up"))
            x = x + (gate / (1 + torch.exp(-gate)) * up) @ w[p + "mlp.down_proj.weight"].T
        x = norm(x if rows else x[-1:], w["model.norm.weight"])
        return x @ self.head.T

    def present(self):
        return {"key": self.kv[-1][0], "value": self.kv[-1][1]}


def exact(case, seed):
    k = case["kind"]
    if k == "prefill":
        m = _Exact(case, seed)
        logits = m.forward(_ids(seed, case["seq"]))[0]
        return {"logits": logits, "argmax": None, "present": m.present()}
    if k == "score":
        m, ids = _Exact(case, seed), _ids(seed, case["seq"])
        lp = torch.log_softmax(m.forward(ids[:-1], rows=True), 1)
        nll = -lp[torch.arange(len(ids) - 1, device="cuda"), torch.from_numpy(ids[1:].astype(np.int64)).cuda()]
        return {"nll": nll, "present": m.present()}
    if k == "decode":
        m = _Exact(case, seed)
        logits = m.forward(_ids(seed, case["ctx"]))
        for _ in range(case["steps"]):
            top = torch.topk(logits[0], 2)
            if float(top.values[0] - top.values[1]) < 2e-3:
                return None  # the greedy choice is within the arithmetic's own error
            logits = m.forward([int(top.indices[0])])
        return {"tokens": None, "logits": logits[0]}
    t = _inputs(case, seed)
    d = {n: x.double() for n, x in t.items() if x is not None and x.is_floating_point()}
    if k == "glue":
        n = case["rows"]
        norm = d["x"] / torch.sqrt((d["x"] ** 2).mean(1, keepdim=True) + CFG.eps) * d["gain"]
        cos, sin = (c.float().double()[n:, None] for c in _rope_tables(2 * n))
        q = d["q"].reshape(n, CFG.heads, HD)
        q = torch.cat((q[..., :32] * cos - q[..., 32:] * sin, q[..., 32:] * cos + q[..., :32] * sin), 2).reshape(n, HIDDEN)
        keys = torch.zeros((CFG.kv_heads, 2 * n, HD), dtype=torch.float64, device="cuda")
        values = torch.zeros((CFG.kv_heads, HD, (2 * n + 63) // 64 * 64), dtype=torch.float64, device="cuda")
        keys[:, n:] = t["k"].half().double().reshape(n, CFG.kv_heads, HD).transpose(0, 1)
        values[:, :, n:2 * n] = t["v"].half().double().reshape(n, CFG.kv_heads, HD).permute(1, 2, 0)
        return {"norm": norm, "q": q, "gate": d["gate"] / (1 + torch.exp(-d["gate"])) * d["up"],
                "x": d["x"] + d["delta"], "keys": keys, "values": values}
    if k in ("matvec", "matmul"):
        return {"y": d["x"] @ _dequantize(t["q"], t["s"], t["z"], case["fmt"]).T + d["b"]}
    if k == "list":
        y = torch.empty((case["count"], case["rows"]), dtype=torch.float64, device="cuda")
        for i in range(case["count"]):
            y[i] = _dequantize(t["q"][i], t["s"][i], None, "int8") @ d["x"][i]
        return {"y": y}
    if k == "attn":
        total, seq = _total(case), case.get("seq", 1)
        q = d["q"].reshape(seq, case["heads"], HD)
        out = [_attend(q, t["k"][i].double(), t["v"][i, :, :, :total].double().transpose(1, 2).contiguous(), total - seq)
               for i in range(case.get("count", 1))]
        return {"out": torch.cat(out).reshape(-1, case["heads"] * HD)}
    q, s, z = _quantize(t["w"].float(), case["to"])
    out = {"data": q.double() if case["to"] == "f16" else q}
    if s is not None:
        out["scales"] = s
    if z is not None:
        out["zeros"] = z
    return out
