"""The workloads whose speed is tracked: what programs built on tang_amd run,
through its public entry points (capi and the C ABI behind it).

Every case has a "kind" (the path), sizes and data types.  `listed()` names a
fixed set, `draw()` gives further cases of the same ranges, `prepare()` makes
what a program has in hand before the call (inputs from the seed, weights,
output buffers, recorded graphs), `run()` is one pass, `exact()` the same
outputs from plain torch in 64 bits.  Decode-sized sequences of calls are
recorded once with capture() and replayed, as the decode loops of such
programs do; prefill-sized ones are enqueued call by call.
"""
import concurrent.futures
import ctypes
import math

import numpy as np
import torch

from tang_amd import capi

# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------


def listed():
    return [
        # One decode token's int4 linears (QKV, O, gate/up, down of two
        # 7B-shaped layers) at batch 1: the weight-streaming GEMV.
        dict(name="q4_decode", kind="q4", m=1, layers=2, d=4096, kv=4096, ff=11008, x="bf16", scales="f16", graph=True),
        # Thirteen sequences decoded together with reference-quantized blocks
        # (f32 scales), f32 activations and widths that fill neither a
        # 32-group nor a tile.
        dict(name="q4_batch", kind="q4", m=13, layers=2, d=2500, kv=500, ff=6700, x="f32", scales="f32", graph=True),
        # A 2048-token prompt through one 7B-shaped layer's linears.
        dict(name="q4_prefill", kind="q4", m=2048, layers=1, d=4096, kv=4096, ff=11008, x="bf16", scales="f16",
             graph=False),
        # int8 per-row GEMV at batch 1 (4096 x 4096), eight layers' matrices.
        dict(name="q8_decode", kind="q8", m=1, rows=4096, cols=4096, copies=8, scales="row", x="f32", graph=True),
        # A batch of 100 rows through an int8 matrix with per-block scales
        # (quantize_matrix_q8 output).
        dict(name="q8_batch", kind="q8", m=100, rows=11008, cols=4096, copies=1, scales="group", x="bf16",
             graph=False),
        # Unquantized linear (a head kept in bf16) over a prompt chunk, f32
        # activations: matmul_b_transposed.
        dict(name="dense_linear", kind="dense", m=509, k=2048, n=5632, ta=False, tb=True, a="f32", b="bf16"),
        # KV-cached attention of one new token over an 8K context, grouped
        # heads, f16 cache, four layers.
        dict(name="attn_decode", kind="attn", q_len=1, start=8191, heads=32, kv_heads=8, hd=128, cache="f16",
             layers=4, graph=True),
        # A transformer block composed op by op (norm, QKV, RoPE, cache
        # append, attention, O, residual norm, SwiGLU MLP) for a 384-token
        # prompt chunk behind 512 cached positions.
        dict(name="block_prefill", kind="block", T=384, start=512, d=2048, heads=16, kv_heads=8, hd=128, ff=5632),
        # Mixture-of-experts layer (64 + 2 int4 experts, top-6), decode batch.
        dict(name="moe_decode", kind="moe", T=16, d=2048, ff=1408, E=64, S=2, k=6),
        # The same layer for a prompt chunk.
        dict(name="moe_prefill", kind="moe", T=512, d=2048, ff=1408, E=64, S=2, k=6),
        # Latent-attention decode, eight sequences of 4096 cached positions.
        dict(name="mla_decode", kind="mla", B=8, L=4096, dn=128, dr=64, r=512, dv=128),
        # The decode engine as a program drives it with its own sampling:
        # a prompt, then token by token with the logits read each step.
        dict(name="llama_chat", kind="llama", n=450, steps=8, n_layers=4, d=2048, heads=16, kv_heads=8, hd=128, ff=5632,
             vocab=32000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["q4", "q4", "q4", "q8", "q8", "dense", "attn", "attn", "block", "moe", "mla", "llama"])
    if kind == "q4":
        d = rng.choice([1024, 2048, 4096, rng.randrange(600, 4096), 8 * rng.randrange(100, 512)])
        ff = rng.choice([2752, 5632, 11008, rng.randrange(1500, 11008), 8 * rng.randrange(200, 1376)])
        m = _log_int(rng, 1, 2048)
        return dict(kind=kind, m=m, layers=2 if m <= 64 else 1, d=d, kv=rng.choice([d, max(8, d // 4 // 8 * 8)]), ff=ff,
                    x=rng.choice(["bf16", "f32"]), scales=rng.choice(["f16", "f16", "f32"]), graph=m <= 16)
    if kind == "q8":
        m = _log_int(rng, 1, 256)
        return dict(kind=kind, m=m, rows=rng.choice([2048, 4096, 11008, rng.randrange(500, 11008)]),
                    cols=rng.choice([2048, 4096, 8 * rng.randrange(64, 1024), rng.randrange(500, 8192)]),
                    copies=4 if m <= 8 else 1, scales=rng.choice(["row", "group"]), x=rng.choice(["bf16", "f32"]),
                    graph=m <= 8)
    if kind == "dense":
        return dict(kind=kind, m=_log_int(rng, 1, 1024), k=rng.choice([576, 2048, 4096, rng.randrange(64, 4096)]),
                    n=rng.choice([64, 1536, 5632, rng.randrange(64, 8192)]), ta=rng.random() < 0.2,
                    tb=rng.random() < 0.7, a=rng.choice(["f32", "f32", "bf16"]), b=rng.choice(["f32", "bf16"]))
    if kind == "attn":
        q_len = rng.choice([1, 1, _log_int(rng, 2, 640)])
        kv_heads = rng.choice([4, 8, 16])
        return dict(kind=kind, q_len=q_len, start=_log_int(rng, 1, 16000 if q_len == 1 else 2048), kv_heads=kv_heads,
                    heads=kv_heads * rng.choice([1, 2, 4]), hd=rng.choice([64, 128, 128, 256]),
                    cache=rng.choice(["f16", "f16", "f32"]), layers=2 if q_len == 1 else 1, graph=q_len == 1)
    if kind == "block":
        kv_heads, hd = rng.choice([4, 8]), rng.choice([64, 128])
        heads = kv_heads * rng.choice([1, 2, 4])
        return dict(kind=kind, T=_log_int(rng, 17, 700), start=rng.randrange(0, 1024), d=heads * hd, heads=heads,
                    kv_heads=kv_heads, hd=hd, ff=8 * rng.randrange(96, 704))
    if kind == "moe":
        d, ff, E, S, k = rng.choice([(2048, 1408, 64, 2, 6), (1024, 704, 32, 1, 4), (256, 96, 8, 1, 3)])
        return dict(kind=kind, T=_log_int(rng, 1, 700), d=d, ff=ff, E=E, S=S, k=k)
    if kind == "mla":
        r, dr = rng.choice([(512, 64), (512, 64), (256, 64), (64, 32)])
        return dict(kind=kind, B=rng.randrange(1, 17), L=_log_int(rng, 16, 4096), dn=rng.choice([128, 64]), dr=dr, r=r,
                    dv=rng.choice([128, 64]))
    kv_heads = rng.choice([2, 4])
    heads = kv_heads * rng.choice([1, 2, 4])
    return dict(kind="llama", n=_log_int(rng, 5, 1100), steps=rng.randrange(2, 12), n_layers=2, d=heads * 128, heads=heads,
                kv_heads=kv_heads, hd=128, ff=8 * rng.randrange(64, 512), vocab=rng.randrange(2000, 16000))


# ---------------------------------------------------------------------------
# Shared pieces
# ---------------------------------------------------------------------------

_dev = None
_models = {}  # kind -> (configuration, model): the one model of each kind a program keeps loaded
_DT = {"f32": capi.F32, "bf16": capi.BF16, "f16": capi.F16}


def _device():
    global _dev
    if _dev is None:
        _dev = capi.HipComputeDevice(0)
    return _dev


class _BufferRecord(ctypes.Structure):
    """The record behind a buffer handle (th_buffer, csrc/common.hpp)."""
    _fields_ = [("dev", ctypes.c_void_p), ("dtype", ctypes.c_int), ("n", ctypes.c_size_t), ("ptr", ctypes.c_void_p)]


class _Span:
    def __init__(self, buf, typestr, shape):
        rec = ctypes.cast(buf.handle, ctypes.POINTER(_BufferRecord)).contents
        self.keep = buf
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, data=(rec.ptr, False), version=2,
                                             strides=None)


def _view(buf, *shape):
    """A torch view of a library buffer (no copy: outputs stay on the GPU)."""
    typestr = {capi.F32: "<f4", capi.F16: "<f2", capi.I32: "<i4"}[buf.dtype]
    return torch.as_tensor(_Span(buf, typestr, shape), device="cuda")


def _bf16_bits(v):
    b = np.ascontiguousarray(v, np.float32).view(np.uint32)
    return ((b + 0x7FFF + ((b >> 16) & 1)) >> 16).astype(np.uint16)


def _host(v, dt):
    """f32 values as the host array a buffer of type dt takes."""
    return _bf16_bits(v) if dt == "bf16" else v.astype(np.float16).view(np.uint16) if dt == "f16" else v


def _wide(bits, dt):
    """Those values, exactly, as a float64 tensor on the GPU."""
    t = torch.from_numpy(bits).cuda() if dt == "f32" else torch.from_numpy(bits.view(np.int16)).cuda()
    if dt == "bf16":
        t = t.view(torch.bfloat16)
    elif dt == "f16":
        t = t.view(torch.float16)
    return t.to(torch.float64)


def _normal(rng, *shape, std=1.0):
    v = rng.standard_normal(shape, dtype=np.float32)
    return v * np.float32(std) if std != 1.0 else v


def _check(rc):
    capi.check(rc)


def _capture(dev, fn):
    """fn's calls recorded for replay (made once before: workspaces grow)."""
    fn()
    dev.sync()
    return dev.capture(fn)


def _q4_host(rng, rows, cols, scales):
    bpr = (cols + 31) // 32
    nib = np.frombuffer(rng.bytes(rows * bpr * 16), np.uint8).reshape(rows, bpr * 16)
    sc = rng.uniform(0.002, 0.01, (rows, bpr)).astype(np.float16 if scales == "f16" else np.float32)
    return nib, sc.view(np.uint16) if scales == "f16" else sc


def _q4_upload(dev, w, rows, cols, scales):
    return dev.q4_upload_packed(w[0], w[1], rows, cols, _DT[scales])


def _q4_wide(w, rows, cols):
    nib = torch.from_numpy(np.array(w[0])).cuda()
    sc = w[1].view(np.float16) if w[1].dtype == np.uint16 else w[1]
    s = torch.from_numpy(np.array(sc)).cuda().to(torch.float64)
    v = torch.stack(((nib & 15), (nib >> 4)), -1).reshape(rows, -1, 32).to(torch.float64) - 8.0
    return (v * s[:, :, None]).reshape(rows, -1)[:, :cols]


def _q4_bytes(rows, cols, scales):
    bpr = (cols + 31) // 32
    return rows * bpr * (16 + (2 if scales == "f16" else 4))


def _rope_wide(x, start, heads, hd, base=1e4):
    """Interleaved pairs rotated at positions start..; x [T, heads*hd]."""
    T = x.shape[0]
    freq = base ** (-torch.arange(hd // 2, dtype=torch.float64, device=x.device) / (hd // 2))
    ang = (start + torch.arange(T, dtype=torch.float64, device=x.device))[:, None] * freq
    c, s = ang.cos()[:, None, :], ang.sin()[:, None, :]
    p = x.reshape(T, heads, hd // 2, 2)
    return torch.stack((p[..., 0] * c - p[..., 1] * s, p[..., 0] * s + p[..., 1] * c), -1).reshape(T, heads * hd)


def _attention_wide(q, k, v, start, heads, kv_heads, hd):
    T, n = q.shape[0], k.shape[0]
    out = torch.empty_like(q)
    mask = torch.arange(n, device=q.device)[None, :] > start + torch.arange(T, device=q.device)[:, None]
    for h in range(heads):
        g = h // (heads // kv_heads)
        s = (q[:, h * hd:(h + 1) * hd] @ k[:, g * hd:(g + 1) * hd].t().contiguous()) / math.sqrt(hd)
        s = s.masked_fill(mask, -math.inf).softmax(-1)
        out[:, h * hd:(h + 1) * hd] = s @ v[:, g * hd:(g + 1) * hd].contiguous()
    return out


def _norm_wide(x, w, eps=1e-5):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w


def _attended(start, T):
    return sum(start + i + 1 for i in range(T))


# ---------------------------------------------------------------------------
# int4 linears
# ---------------------------------------------------------------------------


def _q4_shapes(c):
    return [(c["d"] + 2 * c["kv"], c["d"]), (c["d"], c["d"]), (2 * c["ff"], c["d"]), (c["d"], c["ff"])] * c["layers"]


def _q4_inputs(c, seed):
    rng = np.random.default_rng(seed)
    xd, xf = (_host(_normal(rng, c["m"], n), c["x"]) for n in (c["d"], c["ff"]))
    return xd, xf, [_q4_host(rng, r, k, c["scales"]) for r, k in _q4_shapes(c)]


class _Q4:
    def __init__(self, c, seed):
        dev = _device()
        xd, xf, ws = _q4_inputs(c, seed)
        self.m = c["m"]
        xd, xf = dev.upload(xd, _DT[c["x"]]), dev.upload(xf, _DT[c["x"]])
        self.calls = []
        for i, ((rows, cols), w) in enumerate(zip(_q4_shapes(c), ws)):
            self.calls.append((xf if i % 4 == 3 else xd, _q4_upload(dev, w, rows, cols, c["scales"]),
                               dev.alloc(c["m"] * rows)))
        self.out = [_view(y, c["m"], w.rows) for _, w, y in self.calls]
        self.graph = _capture(dev, self.enqueue) if c["graph"] else None

    def enqueue(self):
        dev = _device()
        for x, w, y in self.calls:
            dev.gemm_q4(x, self.m, w, y)

    def run(self):
        if self.graph:
            self.graph.launch()
        else:
            self.enqueue()
        return self.out


def _q4_exact(c, seed):
    xd, xf, ws = _q4_inputs(c, seed)
    xd, xf = _wide(xd, c["x"]), _wide(xf, c["x"])
    return [(xf if i % 4 == 3 else xd) @ _q4_wide(w, r, k).t() for i, ((r, k), w) in enumerate(zip(_q4_shapes(c), ws))]


# ---------------------------------------------------------------------------
# int8 linears
# ---------------------------------------------------------------------------


def _q8_inputs(c, seed):
    rng = np.random.default_rng(seed)
    rows, cols = c["rows"], c["cols"]
    x = _host(_normal(rng, c["m"], cols), c["x"])
    ws = []
    for _ in range(c["copies"]):
        q = rng.integers(-127, 128, (rows, cols), np.int8)
        n = 1 if c["scales"] == "row" else (cols + 31) // 32
        ws.append((q, rng.uniform(0.005, 0.02, (rows, n)).astype(np.float32)))
    return x, ws


def _q8_upload(dev, q, s):
    rows, cols = q.shape
    if s.shape[1] == 1:
        return dev.q8_upload_rowwise(q, s.reshape(-1), rows, cols)
    bpr = s.shape[1]
    blocks = np.zeros((rows, bpr), capi.Q8_BLOCK)
    blocks["scale"] = s
    padded = np.zeros((rows, bpr * 32), np.int8)
    padded[:, :cols] = q
    blocks["values"] = padded.reshape(rows, bpr, 32)
    return dev.q8_upload_blocks(blocks.reshape(-1), rows, cols)


class _Q8:
    def __init__(self, c, seed):
        dev = _device()
        x, ws = _q8_inputs(c, seed)
        self.m, self.x = c["m"], dev.upload(x, _DT[c["x"]])
        self.calls = [(_q8_upload(dev, q, s), dev.alloc(c["m"] * c["rows"])) for q, s in ws]
        self.out = [_view(y, c["m"], c["rows"]) for _, y in self.calls]
        self.graph = _capture(dev, self.enqueue) if c["graph"] else None

    def enqueue(self):
        dev = _device()
        for w, y in self.calls:
            dev.gemv_q8(self.x, self.m, w, y)

    def run(self):
        if self.graph:
            self.graph.launch()
        else:
            self.enqueue()
        return self.out


def _q8_exact(c, seed):
    x, ws = _q8_inputs(c, seed)
    x = _wide(x, c["x"])
    out = []
    for q, s in ws:
        w = torch.from_numpy(q).cuda().to(torch.float64)
        s = torch.from_numpy(s).cuda().to(torch.float64)
        w *= s if s.shape[1] == 1 else s.repeat_interleave(32, 1)[:, :q.shape[1]]
        out.append(x @ w.t())
    return out


# ---------------------------------------------------------------------------
# Dense matmul
# ---------------------------------------------------------------------------


def _dense_inputs(c, seed):
    rng = np.random.default_rng(seed)
    m, k, n = c["m"], c["k"], c["n"]
    a = _host(_normal(rng, *((k, m) if c["ta"] else (m, k))), c["a"])
    b = _host(_normal(rng, *((n, k) if c["tb"] else (k, n)), std=1.0 / math.sqrt(k)), c["b"])
    return a, b


class _Dense:
    def __init__(self, c, seed):
        dev = _device()
        a, b = _dense_inputs(c, seed)
        m, k, n = c["m"], c["k"], c["n"]
        self.a, self.b, self.c = dev.upload(a, _DT[c["a"]]), dev.upload(b, _DT[c["b"]]), dev.alloc(m * n)
        self.args = (m, k, n, int(c["ta"]), int(c["tb"]), 0)
        self.out = _view(self.c, m, n)

    def run(self):
        _check(capi.lib().th_matmul_ex(_device().handle, self.a.handle, self.b.handle, *self.args, self.c.handle))
        return self.out


def _dense_exact(c, seed):
    a, b = _dense_inputs(c, seed)
    a, b = _wide(a, c["a"]), _wide(b, c["b"])
    return (a.t().contiguous() if c["ta"] else a) @ (b.t().contiguous() if c["tb"] else b)


# ---------------------------------------------------------------------------
# KV-cached attention
# ---------------------------------------------------------------------------


def _attn_inputs(c, seed):
    rng = np.random.default_rng(seed)
    n, kvd = c["start"] + c["q_len"], c["kv_heads"] * c["hd"]
    return [(_normal(rng, c["q_len"], c["heads"] * c["hd"]), _host(_normal(rng, n, kvd), c["cache"]),
             _host(_normal(rng, n, kvd), c["cache"])) for _ in range(c["layers"])]


class _Attn:
    def __init__(self, c, seed):
        dev = _device()
        self.sizes = (c["start"], c["q_len"], c["heads"], c["kv_heads"], c["hd"])
        dt = _DT[c["cache"]]
        self.calls = [(dev.upload(q), dev.upload(k, dt), dev.upload(v, dt), dev.alloc(q.size))
                      for q, k, v in _attn_inputs(c, seed)]
        self.out = [_view(o, c["q_len"], c["heads"] * c["hd"]) for _, _, _, o in self.calls]
        self.graph = _capture(dev, self.enqueue) if c["graph"] else None

    def enqueue(self):
        L, h = capi.lib(), _device().handle
        for q, k, v, o in self.calls:
            _check(L.th_kv_attention(h, q.handle, k.handle, v.handle, *self.sizes, o.handle))

    def run(self):
        if self.graph:
            self.graph.launch()
        else:
            self.enqueue()
        return self.out


def _attn_exact(c, seed):
    return [_attention_wide(_wide(q, "f32"), _wide(k, c["cache"]), _wide(v, c["cache"]), c["start"], c["heads"],
                            c["kv_heads"], c["hd"]) for q, k, v in _attn_inputs(c, seed)]


# ---------------------------------------------------------------------------
# A transformer block composed from the operators
# ---------------------------------------------------------------------------


def _block_inputs(c, seed):
    rng = np.random.default_rng(seed)
    d, ff, kvd = c["d"], c["ff"], c["kv_heads"] * c["hd"]
    shapes = dict(wq=(d, d), wk=(kvd, d), wv=(kvd, d), wo=(d, d), wg=(ff, d), wu=(ff, d), wd=(d, ff))
    w = {n: _q4_host(rng, r, k, "f16") for n, (r, k) in shapes.items()}
    n1, n2 = (_host(1.0 + _normal(rng, d, std=0.1), "bf16") for _ in range(2))
    x = _normal(rng, c["T"], d)
    rows = c["start"] + c["T"]
    kc, vc = (_host(_normal(rng, rows, kvd), "f16") for _ in range(2))
    return shapes, w, n1, n2, x, kc, vc


class _Block:
    def __init__(self, c, seed):
        dev = _device()
        self.c = c
        T, d, ff, kvd = c["T"], c["d"], c["ff"], c["kv_heads"] * c["hd"]
        shapes, w, n1, n2, x, kc, vc = _block_inputs(c, seed)
        self.w = {n: _q4_upload(dev, w[n], *shapes[n], "f16") for n in w}
        self.n1, self.n2, self.x = dev.upload(n1, capi.BF16), dev.upload(n2, capi.BF16), dev.upload(x)
        self.kc, self.vc = dev.upload(kc, capi.F16), dev.upload(vc, capi.F16)
        cs, sn = capi.rope_tables(c["hd"], c["start"] + T, 1e4)
        self.cs, self.sn = dev.upload(cs), dev.upload(sn)
        sizes = dict(h=d, q=d, k=kvd, v=kvd, qr=d, kr=kvd, a=d, o=d, h2=d, s=d, g=ff, u=ff, act=ff, dn=d, out=d)
        self.b = {n: dev.alloc(T * w_) for n, w_ in sizes.items()}
        self.k16, self.v16 = dev.alloc(T * kvd, capi.F16), dev.alloc(T * kvd, capi.F16)
        self.out = [_view(self.b["out"], T, d), _view(self.kc, c["start"] + T, kvd), _view(self.vc, c["start"] + T, kvd)]

    def run(self):
        c, b, L, dev = self.c, self.b, capi.lib(), _device()
        T, d, ff, kvd, start = c["T"], c["d"], c["ff"], c["kv_heads"] * c["hd"], c["start"]
        h = dev.handle
        H = {n: v.handle for n, v in b.items()}

        def linear(x, w, y):
            dev.gemm_q4(b[x], T, self.w[w], b[y])

        _check(L.th_rms_norm(h, self.x.handle, self.n1.handle, T, d, 1e-5, H["h"]))
        linear("h", "wq", "q")
        linear("h", "wk", "k")
        linear("h", "wv", "v")
        _check(L.th_rope_forward(h, H["q"], self.cs.handle, self.sn.handle, T, c["heads"], c["hd"], start, H["qr"]))
        _check(L.th_rope_forward(h, H["k"], self.cs.handle, self.sn.handle, T, c["kv_heads"], c["hd"], start, H["kr"]))
        _check(L.th_convert(h, H["kr"], self.k16.handle))
        _check(L.th_convert(h, H["v"], self.v16.handle))
        _check(L.th_buffer_copy_region(self.kc.handle, start * kvd, self.k16.handle, 0, T * kvd))
        _check(L.th_buffer_copy_region(self.vc.handle, start * kvd, self.v16.handle, 0, T * kvd))
        _check(L.th_kv_attention(h, H["qr"], self.kc.handle, self.vc.handle, start, T, c["heads"], c["kv_heads"],
                                 c["hd"], H["a"]))
        linear("a", "wo", "o")
        _check(L.th_rms_norm_residual(h, H["o"], self.x.handle, self.n2.handle, T, d, 1e-5, H["h2"], H["s"]))
        linear("h2", "wg", "g")
        linear("h2", "wu", "u")
        _check(L.th_swiglu(h, H["g"], H["u"], T * ff, H["act"]))
        linear("act", "wd", "dn")
        _check(L.th_add(h, H["s"], H["dn"], T * d, H["out"]))
        return self.out


def _block_exact(c, seed):
    T, d, start = c["T"], c["d"], c["start"]
    shapes, w, n1, n2, x, kc, vc = _block_inputs(c, seed)
    W = {n: _q4_wide(w[n], *shapes[n]) for n in w}
    x, n1, n2 = _wide(x, "f32"), _wide(n1, "bf16"), _wide(n2, "bf16")
    kc, vc = _wide(kc, "f16"), _wide(vc, "f16")
    h = _norm_wide(x, n1)
    q = _rope_wide(h @ W["wq"].t(), start, c["heads"], c["hd"])
    kc[start:] = _rope_wide(h @ W["wk"].t(), start, c["kv_heads"], c["hd"])
    vc[start:] = h @ W["wv"].t()
    a = _attention_wide(q, kc, vc, start, c["heads"], c["kv_heads"], c["hd"])
    s = a @ W["wo"].t() + x
    h2 = _norm_wide(s, n2)
    g, u = h2 @ W["wg"].t(), h2 @ W["wu"].t()
    return [(g * g.sigmoid() * u) @ W["wd"].t() + s, kc, vc]


# ---------------------------------------------------------------------------
# Mixture of experts
# ---------------------------------------------------------------------------

_MOE_SEED, _LLAMA_SEED = 4, 3  # the models' weights: loaded once, the same for every input


def _model(kind, config, make, destroy):
    """The loaded model of this kind; another configuration replaces it."""
    have = _models.get(kind)
    if have is None or have[0] != config:
        if have is not None:
            destroy(_models.pop(kind)[1])
        _models[kind] = (config, make())
    return _models[kind][1]


def _moe_make(c):
    L, h = capi.lib(), ctypes.c_void_p()
    _check(L.th_moe_create(_device().handle, c["d"], c["ff"], c["E"], c["S"], c["k"], ctypes.byref(h)))
    _check(L.th_moe_init_synthetic(h, _MOE_SEED))
    return h


def _moe_input(c, seed):
    return _host(_normal(np.random.default_rng(seed), c["T"], c["d"]), "bf16")


class _Moe:
    def __init__(self, c, seed):
        dev = _device()
        self.moe = _model("moe", tuple(c[n] for n in ("d", "ff", "E", "S", "k")), lambda: _moe_make(c),
                          capi.lib().th_moe_destroy)
        self.T, T = c["T"], c["T"]
        self.h = dev.upload(_moe_input(c, seed), capi.BF16)
        self.o, self.i, self.w = dev.alloc(T * c["d"]), dev.alloc(T * c["k"], capi.I32), dev.alloc(T * c["k"])
        self.out = [_view(self.o, T, c["d"]), _view(self.i, T, c["k"]), _view(self.w, T, c["k"])]

    def run(self):
        _check(capi.lib().th_moe_forward(self.moe, self.h.handle, self.T, self.o.handle, self.i.handle, self.w.handle))
        return self.out


def _moe_exact(c, seed):
    d, ff, E, S, k, T = (c[n] for n in ("d", "ff", "E", "S", "k", "T"))
    h = _wide(_moe_input(c, seed), "bf16")
    wr = torch.from_numpy(capi.synth_normal(capi.synth_seed(_MOE_SEED, 1000, 0), E * d, 0.02)).cuda().double()
    p = (h @ wr.reshape(E, d).t()).softmax(-1)
    w, idx = p.topk(k, -1)
    out = torch.zeros(T, d, dtype=torch.float64, device="cuda")
    shapes = ((4, ff, d), (5, ff, d), (6, d, ff))
    with concurrent.futures.ThreadPoolExecutor(8) as pool:  # the layer's weights, as it was filled with them
        made = pool.map(lambda e: [capi.synth_q4(capi.synth_seed(_MOE_SEED, e, t), r, n) for t, r, n in shapes],
                        range(E + S))
        for e, ws in enumerate(made):
            tok, rank = (idx == e).nonzero(as_tuple=True) if e < E else (torch.arange(T, device="cuda"), None)
            if not len(tok):
                continue
            g, u, dn = (_q4_wide(w_, r, n) for w_, (_, r, n) in zip(ws, shapes))
            x = h[tok]
            gx = x @ g.t()
            y = (gx * gx.sigmoid() * (x @ u.t())) @ dn.t()
            out.index_add_(0, tok, y if rank is None else y * w[tok, rank][:, None])
    return [out, idx.to(torch.int32), w]


# ---------------------------------------------------------------------------
# Latent attention
# ---------------------------------------------------------------------------


def _mla_inputs(c, seed):
    rng = np.random.default_rng(seed)
    B, L, dn, dr, r, dv = (c[n] for n in ("B", "L", "dn", "dr", "r", "dv"))
    qn, qr = _normal(rng, B, 16, dn), _normal(rng, B, 16, dr)
    cache = _host(_normal(rng, B, L, r + dr), "bf16")
    uk, uv = rng.integers(-127, 128, (16 * r, dn), np.int8), rng.integers(-127, 128, (16 * dv, r), np.int8)
    sk, sv = (rng.uniform(0.0005, 0.002, n).astype(np.float32) for n in (16 * r, 16 * dv))
    return qn, qr, cache, uk, sk, uv, sv


class _Mla:
    def __init__(self, c, seed):
        dev = _device()
        qn, qr, cache, uk, sk, uv, sv = _mla_inputs(c, seed)
        self.qn, self.qr, self.cache = dev.upload(qn), dev.upload(qr), dev.upload(cache, capi.BF16)
        self.uk, self.uv = dev.q8_upload_rowwise(uk, sk, *uk.shape), dev.q8_upload_rowwise(uv, sv, *uv.shape)
        self.sizes = (c["B"], 16, c["L"], c["dn"], c["dr"], c["r"], c["dv"])
        self.scale = 1.0 / math.sqrt(c["dn"] + c["dr"])
        self.o = dev.alloc(c["B"] * 16 * c["dv"])
        self.out = _view(self.o, c["B"], 16, c["dv"])

    def run(self):
        _device().mla_decode(self.qn, self.qr, self.cache, *self.sizes, self.uk, self.uv, self.scale, self.o)
        return self.out


def _mla_exact(c, seed):
    B, L, dn, dr, r, dv = (c[n] for n in ("B", "L", "dn", "dr", "r", "dv"))
    qn, qr, cache, uk, sk, uv, sv = _mla_inputs(c, seed)
    uk = torch.from_numpy(uk).cuda().double() * torch.from_numpy(sk).cuda().double()[:, None]
    uv = torch.from_numpy(uv).cuda().double() * torch.from_numpy(sv).cuda().double()[:, None]
    uk, uv = uk.reshape(16, r, dn), uv.reshape(16, dv, r)
    qn, qr, cache = _wide(qn, "f32"), _wide(qr, "f32"), _wide(cache, "bf16")
    out = torch.empty(B, 16, dv, dtype=torch.float64, device="cuda")
    for b in range(B):
        lat = torch.stack([uk[h] @ qn[b, h] for h in range(16)])
        s = torch.cat((lat, qr[b]), 1) @ cache[b].t().contiguous() / math.sqrt(dn + dr)
        o = s.softmax(-1) @ cache[b, :, :r].contiguous()
        out[b] = torch.stack([uv[h] @ o[h] for h in range(16)])
    return out


# ---------------------------------------------------------------------------
# The decode engine
# ---------------------------------------------------------------------------


def _llama_config(c):
    rows = -(-(c["n"] + c["steps"] + 1) // 64) * 64
    return capi.LlamaConfig(c["n_layers"], c["d"], c["heads"], c["kv_heads"], c["hd"], c["ff"], c["vocab"], rows, 1e-5,
                            1e4)


def _llama_make(c):
    L, h = capi.lib(), ctypes.c_void_p()
    _check(L.th_llama_create(_device().handle, ctypes.byref(_llama_config(c)), ctypes.byref(h)))
    _check(L.th_llama_init_synthetic(h, _LLAMA_SEED))
    return h


def _llama_tokens(c, seed):
    rng = np.random.default_rng(seed)
    return rng.integers(0, c["vocab"], c["n"] + c["steps"], np.int32)


class _Llama:
    def __init__(self, c, seed):
        cfg = tuple(c[n] for n in ("n", "steps", "n_layers", "d", "heads", "kv_heads", "hd", "ff", "vocab"))
        self.model = _model("llama", cfg, lambda: _llama_make(c), capi.lib().th_llama_destroy)
        self.c, self.tokens = c, _llama_tokens(c, seed)

    def run(self):
        c, L, t = self.c, capi.lib(), self.tokens
        logits = np.empty((c["steps"] + 1, c["vocab"]), np.float32)
        greedy = np.empty(1, np.int32)
        _check(L.th_llama_prefill(self.model, capi.ptr(t), c["n"], 0, capi.ptr(greedy), capi.ptr(logits[0])))
        for i in range(c["steps"]):  # the program's own choice of token goes in at every step
            _check(L.th_llama_generate(self.model, int(t[c["n"] + i]), c["n"] + i, 1, capi.ptr(greedy),
                                       capi.ptr(logits[i + 1])))
        return logits


def _llama_exact(c, seed):
    L, d, ff, V, hd = c["n_layers"], c["d"], c["ff"], c["vocab"], c["hd"]
    qd, kvd = c["heads"] * hd, c["kv_heads"] * hd
    t = torch.from_numpy(_llama_tokens(c, seed).astype(np.int64)).cuda()

    def linear(layer, tensor, rows, cols):  # the weights the engine was filled with
        return _q4_wide(capi.synth_q4(capi.synth_seed(_LLAMA_SEED, layer, tensor), rows, cols), rows, cols).t()

    def vector(layer, tensor, n):
        return _wide(capi.synth_normal(capi.synth_seed(_LLAMA_SEED, layer, tensor), n, 0.02, capi.BF16), "bf16")

    x = vector(L, 10, V * d).reshape(V, d)[t]
    for l in range(L):
        h = _norm_wide(x, vector(l, 7, d))
        q = _rope_wide(h @ linear(l, 0, qd, d), 0, c["heads"], hd)
        k = _rope_wide(h @ linear(l, 1, kvd, d), 0, c["kv_heads"], hd)
        x = x + _attention_wide(q, k, h @ linear(l, 2, kvd, d), 0, c["heads"], c["kv_heads"], hd) @ linear(l, 3, d, qd)
        h = _norm_wide(x, vector(l, 8, d))
        g = h @ linear(l, 4, ff, d)
        x = x + (g * g.sigmoid() * (h @ linear(l, 5, ff, d))) @ linear(l, 6, d, ff)
    return _norm_wide(x[c["n"] - 1:], vector(L, 11, d)) @ linear(L, 12, V, d)


# ---------------------------------------------------------------------------
# What the measurement calls
# ---------------------------------------------------------------------------

_STATE = {"q4": _Q4, "q8": _Q8, "dense": _Dense, "attn": _Attn, "block": _Block, "moe": _Moe, "mla": _Mla,
          "llama": _Llama}
_EXACT = {"q4": _q4_exact, "q8": _q8_exact, "dense": _dense_exact, "attn": _attn_exact, "block": _block_exact,
          "moe": _moe_exact, "mla": _mla_exact, "llama": _llama_exact}


def prepare(case, seed):
    return _STATE[case["kind"]](case, seed)


def run(state):
    return state.run()


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def work(case):
    c, kind = case, case["kind"]
    if kind == "q4":
        es = 2 if c["x"] == "bf16" else 4
        shapes = _q4_shapes(c)
        return dict(bytes=sum(_q4_bytes(r, k, c["scales"]) + 4 * c["m"] * r for r, k in shapes) +
                    es * c["m"] * (c["d"] + c["ff"]), flops=sum(2 * c["m"] * r * k for r, k in shapes))
    if kind == "q8":
        es = 2 if c["x"] == "bf16" else 4
        n = 1 if c["scales"] == "row" else (c["cols"] + 31) // 32
        return dict(bytes=c["copies"] * (c["rows"] * (c["cols"] + 4 * n) + 4 * c["m"] * c["rows"]) + es * c["m"] * c["cols"],
                    flops=2 * c["copies"] * c["m"] * c["rows"] * c["cols"])
    if kind == "dense":
        size = {"f32": 4, "bf16": 2}
        m, k, n = c["m"], c["k"], c["n"]
        return dict(bytes=m * k * size[c["a"]] + k * n * size[c["b"]] + 4 * m * n, flops=2 * m * k * n)
    if kind == "attn":
        es, qd = 2 if c["cache"] == "f16" else 4, c["heads"] * c["hd"]
        return dict(bytes=c["layers"] * ((c["start"] + c["q_len"]) * c["kv_heads"] * c["hd"] * 2 * es + 8 * c["q_len"] * qd),
                    flops=c["layers"] * 4 * qd * _attended(c["start"], c["q_len"]))
    if kind == "block":
        d, ff, T, kvd = c["d"], c["ff"], c["T"], c["kv_heads"] * c["hd"]
        lin = 2 * d * d + 2 * kvd * d + 3 * d * ff
        return dict(bytes=lin * 9 // 16 + 8 * T * d + 4 * (c["start"] + 2 * T) * kvd,
                    flops=2 * T * lin + 4 * d * _attended(c["start"], T))
    if kind == "moe":
        d, ff, E, S, k, T = (c[n] for n in ("d", "ff", "E", "S", "k", "T"))
        used = S + E * (1.0 - (1.0 - k / E) ** T)  # experts that T tokens reach
        return dict(bytes=used * 3 * d * ff * 9 / 16 + 4 * E * d + T * (6 * d + 8 * k),
                    flops=6 * T * (k + S) * d * ff + 2 * T * E * d)
    if kind == "mla":
        B, L, dn, dr, r, dv = (c[n] for n in ("B", "L", "dn", "dr", "r", "dv"))
        return dict(bytes=2 * B * L * (r + dr) + 16 * (r * (dn + 4) + dv * (r + 4)) + 64 * B * (dn + dr + dv),
                    flops=2 * 16 * B * (r * dn + L * (2 * r + dr) + r * dv))
    d, ff, n, kvd = c["d"], c["ff"], c["n"], c["kv_heads"] * c["hd"]
    lin = c["n_layers"] * (2 * d * d + 2 * kvd * d + 3 * d * ff)
    head = c["vocab"] * d
    rows = n + c["steps"]
    kv = c["n_layers"] * 4 * kvd  # bytes of K and V a position
    return dict(bytes=(1 + c["steps"]) * (lin + head) * 9 // 16 + kv * (rows + _attended(n, c["steps"])) +
                2 * d * rows + 4 * (1 + c["steps"]) * c["vocab"],
                flops=2 * rows * lin + 2 * (1 + c["steps"]) * head + 4 * d * c["n_layers"] * _attended(0, rows))


# About four times the distance from exact() at which the paths stand: f16
# operands of the int4 GEMM 3.5e-4, the f32-accumulated paths 1e-7 to 1e-6,
# the latent attention's bf16-pair operands 5e-6, a block of int4 GEMMs 5e-4,
# bf16 intermediates of the experts 1.6e-3 and of the engine 2.7e-3.
_TOLERANCE = {
    "q4": dict(rel=1.5e-3, max=1e-2),
    "q8": dict(rel=2e-6, max=2e-5),
    "dense": dict(rel=4e-6, max=4e-5),
    "attn": dict(rel=4e-6, max=4e-5),
    "block": dict(rel=2e-3, max=2e-2),
    "moe": dict(rel=7e-3, max=0.1, differ=0.005),
    "mla": dict(rel=2e-5, max=2e-4),
    "llama": dict(rel=1e-2, max=0.1),
}


def tolerance(case):
    return dict(_TOLERANCE[case["kind"]])
