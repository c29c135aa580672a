"""The work that programs have this library do, as cases that can be timed and checked one by one.

Six kinds, each through the C entry points that a program calls:

  gemv     one quantized row times one matrix: k_quantize and k_matmul_q8.
  decode   one token through one decoder layer (embedding row, RMSNorm, QKV, RoPE, K/V store, attention over the cache,
           Wo + residual, RMSNorm, SwiGLU, W2 + residual), the calls captured once into a graph and replayed. W8A8,
           W8A32 and FP32 weights.
  batch    one token each of several sequences through a layer's matrices (the attention is per sequence and stays
           out): the GEMM entry points on a few rows, captured and replayed likewise.
  prefill  the rows of a prompt through one decoder layer's calls. Q8_0, BF16 and FP32 weights.
  layer    the same for Q8_0 as engine_forward_batch makes them, each call's rows the next one's input.
  engine   a checkpoint loaded by engine_load_context: a prompt's last logits, then the logits of further tokens.

In batch and prefill the products behind the first get rows of their own (the attention's, the second norm's and the
gate's), so that each is held to its own rounding: along a chain of quantized rows one rounding tie turns the next
rows' ties, and the last rows of two correct implementations differ by percents. layer and engine are such chains.

Outputs are the residual rows with the K/V caches and what else the calls compute, or the logits. exact() gives the
same in float64, with the library's own rounding of inputs (Q8_0 activations, BF16 rows) and none of its code.
"""
import ctypes
import os
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "llama3.x.c_amd"))

import llama_hip as lh  # noqa: E402
from llama_hip import checkpoint  # noqa: E402

EPS = 1e-5
TABLE_ROWS = 1024  # rows of the embedding table in the layer cases
VOCAB = 32768      # of the engine cases

# Decoder shapes: the Llama 3 sizes that the benchmark and the tests run.
SHAPES = {
    "1b": {"dim": 2048, "hidden": 8192, "heads": 32, "kv_heads": 8},
    "3b": {"dim": 3072, "hidden": 8192, "heads": 24, "kv_heads": 8},
    "8b": {"dim": 4096, "hidden": 14336, "heads": 32, "kv_heads": 8},
}


def listed():
    def layer(name, kind, shape, dtype, rows, pos):
        return {"name": name, "kind": kind, "dtype": dtype, "rows": rows, "pos": pos, "gs": 64, **SHAPES[shape]}

    return [
        # the smallest call: one 2048 x 2048 matrix and one row, the launch and its latency
        {"name": "gemv_2048", "kind": "gemv", "dtype": "q8", "n": 2048, "d": 2048, "gs": 64},
        # a token of a small chat model, early in its context
        layer("decode_1b", "decode", "1b", "q8", 1, 511),
        # the headline decode: a token at the end of a 2048-token context
        layer("decode_8b", "decode", "8b", "q8", 1, 2047),
        # LLAMA_Q8_ACTIVATIONS=fp32: Q8_0 weights, FP32 activations
        layer("decode_8b_w8a32", "decode", "8b", "w8a32", 1, 700),
        # the FP32 executable's decode
        layer("decode_3b_f32", "decode", "3b", "f32", 1, 300),
        # a few sequences decoded together, and a server's full batch
        layer("batch4_8b", "batch", "8b", "q8", 4, 0),
        layer("batch27_8b", "batch", "8b", "q8", 27, 0),
        # one of the reference's default 256-row prefill batches, late in a prompt
        layer("prefill_8b_256", "prefill", "8b", "q8", 256, 1792),
        # the headline prefill: a 2048-token prompt in one batch
        layer("layer_8b_2048", "layer", "8b", "q8", 2048, 0),
        # LLAMA_PRECISION=bf16, a 512-token prompt
        layer("prefill_3b_bf16", "prefill", "3b", "bf16", 512, 0),
        # the FP32 executable's prefill, a ragged prompt
        layer("prefill_3b_f32", "prefill", "3b", "f32", 333, 0),
        # a whole model: a 600-token prompt, then eight tokens
        {"name": "engine_1b", "kind": "engine", "dtype": "q8", "layers": 2, "rows": 600, "steps": 8, "gs": 64,
         **SHAPES["1b"]},
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(low * (high / low) ** rng.random()))))


def draw(rng):
    kind = rng.choice(("gemv", "decode", "decode", "batch", "batch", "prefill", "prefill", "layer", "engine"))
    gs = rng.choice((64, 64, 64, 64, 64, 128))
    if kind == "gemv":
        return {"kind": kind, "dtype": "q8", "n": gs * _log_int(rng, 8, 14336 // gs), "d": _log_int(rng, 500, 14336),
                "gs": gs}
    shape = dict(SHAPES[rng.choice(("1b", "3b", "8b"))])
    if rng.random() < 0.4:  # a generic decoder: other head groups, a hidden size off the tiles
        hd = rng.choice((64, 128))
        kv = rng.choice((2, 4, 8))
        heads = kv * rng.choice((1, 2, 3, 4))
        while heads * hd < 512:
            heads, kv = 2 * heads, 2 * kv
        shape = {"dim": heads * hd, "hidden": 128 * rng.randint(heads * hd // 64, heads * hd // 32), "heads": heads,
                 "kv_heads": kv}
    if kind == "engine":
        shape["hidden"] = min(shape["hidden"], 8192)
        return {"kind": kind, "dtype": "q8", "layers": rng.randint(1, 2), "rows": _log_int(rng, 2, 600),
                "steps": rng.randint(1, 8), "gs": gs, **shape}
    case = {"kind": kind, "dtype": "q8", "rows": 1, "pos": 0, "gs": gs, **shape}
    if kind == "decode":
        case["dtype"] = rng.choice(("q8", "q8", "q8", "w8a32", "f32"))
        case["pos"] = _log_int(rng, 1, 4000)
    elif kind == "batch":
        case["rows"] = rng.randint(2, 32)
    else:
        case["dtype"] = rng.choice(("q8", "q8", "bf16", "f32")) if kind == "prefill" else "q8"
        most = {"q8": 2048, "bf16": 1024, "f32": 400}[case["dtype"]]
        case["rows"] = _log_int(rng, 2, most)
        case["pos"] = rng.choice((0, 0, _log_int(rng, 1, 4096) - 1 if case["rows"] <= 512 else 0))
    return case


# ---- inputs ------------------------------------------------------------------------------------------------------


def _matrices(c):
    """The layer's matrices as (rows, columns)."""
    d, h, kv = c["dim"], c["hidden"], c["dim"] // c["heads"] * c["kv_heads"]
    return {"wq": (d, d), "wk": (kv, d), "wv": (kv, d), "wo": (d, d), "w1": (h, d), "w3": (h, d), "w2": (d, h)}


def _quantize(x, gs):
    """Q8_0 of rows in groups of gs along the last axis: scale = max|x| / 127, q = round half away from zero, in x's own
    type. Returns (q, scales) in that type."""
    g = x.reshape(*x.shape[:-1], -1, gs)
    s = g.abs().amax(-1) / 127.0
    r = g / torch.where(s > 0, s, torch.ones_like(s))[..., None]
    q = torch.sign(r) * torch.floor(r.abs() + 0.5)
    return q.reshape(x.shape), s


def _seq_len(c):
    n = 512
    while n < c["pos"] + c["rows"]:
        n *= 2
    return n


def _inputs(c, seed):
    """A layer's weights, embedding table, norms, caches, RoPE table and token ids from the seed: FP32 (or the float32
    values of the BF16 weights), or (int8, scales) pairs for Q8_0. Weights ~N(0, 0.02), activations ~N(0, 1)."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(*shape, std=1.0):
        return torch.randn(*shape, generator=g, device="cuda") * std

    q8 = c["dtype"] in ("q8", "w8a32")
    hd = c["dim"] // c["heads"]

    def weight(rows, cols, std):
        w = normal(rows, cols, std=std)
        if not q8:
            return w.bfloat16().float() if c["dtype"] == "bf16" else w
        q, s = _quantize(w, c["gs"])
        return q.to(torch.int8), s.contiguous()

    t = {name: weight(rows, cols, 0.02) for name, (rows, cols) in _matrices(c).items()}
    t["table"] = weight(TABLE_ROWS, c["dim"], 1.0)
    for name in ("norm_att", "norm_ffn"):
        t[name] = 1.0 + normal(c["dim"], std=0.1)
    seq, kv = _seq_len(c), hd * c["kv_heads"]
    # head-major caches: position p of KV head h at h * seq * hd + p * hd; the positions before pos are filled
    for name in ("key", "value"):
        cache = torch.zeros(c["kv_heads"], seq, hd, device="cuda")
        cache[:, :c["pos"]] = normal(c["kv_heads"], c["pos"], hd)
        t[name] = cache
    if c["kind"] in ("batch", "prefill"):
        t["att"], t["mid"] = normal(c["rows"], c["dim"]), normal(c["rows"], c["dim"])
        gate = normal(c["rows"], c["hidden"])
        t["gated"] = torch.nn.functional.silu(gate) * normal(c["rows"], c["hidden"])
    # one row per position: the cosines, each pair's twice, then -sin and +sin (theta 500000)
    p = np.arange(c["pos"], c["pos"] + c["rows"], dtype=np.float64)[:, None]
    angle = p * 500000.0 ** (-np.arange(0, hd, 2, dtype=np.float64) / hd)
    cos, sin = np.repeat(np.cos(angle), 2, 1), np.stack((-np.sin(angle), np.sin(angle)), -1).reshape(len(p), hd)
    t["rope"] = torch.from_numpy(np.concatenate((cos, sin), 1).astype(np.float32)).cuda()
    t["ids"] = torch.randint(0, TABLE_ROWS, (c["rows"],), generator=g, device="cuda", dtype=torch.int32)
    return t, kv, seq


# ---- states ------------------------------------------------------------------------------------------------------


class State:
    """What a program keeps: buffers, the calls to make in order, and a graph or a loaded model."""

    def __init__(self):
        self.lib = lh.load()
        if self.lib.llhip_init() != 0:
            raise RuntimeError("no usable device: %s" % lh.last_error())
        self.lib.kernels_kv_layout_select(b"head")
        self.keep = []       # tensors and argument structs that the calls point into
        self.calls = []      # (function, arguments)
        self.graph = None
        self.model = None
        self.panel = None
        self.out = None

    def call(self, name, *args):
        fn = getattr(self.lib, name)
        self.calls.append((fn, tuple(lh.ptr(a) if hasattr(a, "data_ptr") else a for a in args)))
        self.keep.append(args)

    def make(self):
        for fn, args in self.calls:
            fn(*args)

    def capture(self):
        torch.cuda.synchronize()
        self.make()  # once as plain calls: the library sizes its workspaces on a first call, which no capture may
        torch.cuda.synchronize()
        self.lib.llhip_graph_begin()
        self.make()
        self.graph = self.lib.llhip_graph_end()
        if not self.graph:
            raise RuntimeError("capturing the calls failed")

    def __del__(self):
        if self.graph:
            self.lib.llhip_graph_destroy(self.graph)
        if self.panel is not None:
            self.lib.aligned_buffer_free(ctypes.byref(self.panel))
        if self.model is not None:
            self.lib.engine_free(ctypes.byref(self.model))


def _empty(*shape, dtype=torch.float32):
    return torch.zeros(*shape, device="cuda", dtype=dtype)


def prepare(case, seed):
    state = {"gemv": _prepare_gemv, "decode": _prepare_decode, "batch": _prepare_rows, "prefill": _prepare_rows,
             "layer": _prepare_rows, "engine": _prepare_engine}[case["kind"]](case, seed)
    torch.cuda.synchronize()  # the inputs were made on torch's stream; the library has its own
    return state


def _gemv_inputs(c, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    q, s = _quantize(torch.randn(c["d"], c["n"], generator=g, device="cuda") * 0.02, c["gs"])
    return torch.randn(c["n"], generator=g, device="cuda"), q.to(torch.int8), s.contiguous()


def _prepare_gemv(c, seed):
    st = State()
    x, wq, ws = _gemv_inputs(c, seed)
    xq, xs = _empty(c["n"], dtype=torch.int8), _empty(c["n"] // c["gs"])
    y = _empty(c["d"])
    st.call("k_quantize", xq, xs, x, c["n"], c["gs"])
    st.call("k_matmul_q8", y, lh.k8(xq, xs), lh.w8(wq, ws), c["n"], c["d"], c["gs"])
    st.keep.append((xq, xs, wq, ws))
    st.out = y
    return st


def _prepare_decode(c, seed):
    """The engine's decode calls of one layer (one row), captured."""
    st = State()
    t, kv, seq = _inputs(c, seed)
    st.keep.append(t)
    d, h, nh, nkv, gs, pos = c["dim"], c["hidden"], c["heads"], c["kv_heads"], c["gs"], c["pos"]
    hd = d // nh
    x, xb, q, k, v, hb = _empty(d), _empty(d), _empty(d), _empty(kv), _empty(kv), _empty(h)
    xq, xs, hq, hs = _empty(d, dtype=torch.int8), _empty(d // gs), _empty(h, dtype=torch.int8), _empty(h // gs)
    st.keep.append((x, xb, q, k, v, hb, xq, xs, hq, hs))
    dtype = c["dtype"]
    if dtype == "f32":
        st.call("k_embed_f32_rows", x, t["table"], t["ids"], 1, d, TABLE_ROWS)
    else:
        st.call("k_embed_q8_rows", x, t["table"][0], t["table"][1], t["ids"], 1, d, gs, TABLE_ROWS)
    in_d = lh.k8(None, None, xb) if dtype == "w8a32" else lh.k8(xq, xs)
    in_h = lh.k8(None, None, hb) if dtype == "w8a32" else lh.k8(hq, hs)

    def w(name):
        return t[name] if dtype == "f32" else lh.w8(*t[name])

    def quantize(qq, ss, src, n):
        if dtype == "q8":
            st.call("k_quantize", qq, ss, src, n, gs)

    st.call("k_rmsnorm", xb, x, t["norm_att"], d, EPS)
    quantize(xq, xs, xb, d)
    if dtype == "f32":
        st.call("k_matmul_qkv", q, k, v, xb, w("wq"), w("wk"), w("wv"), d, d, kv)
    else:
        st.call("k_matmul_q8_qkv", q, k, v, in_d, w("wq"), w("wk"), w("wv"), d, d, kv, gs)
    st.call("k_rope_apply", q, k, t["rope"], nh, nkv, hd)
    st.call("k_kv_store", t["key"], k, kv, pos, 1, nkv, hd, seq)
    st.call("k_kv_store", t["value"], v, kv, pos, 1, nkv, hd, seq)
    st.call("k_attention_kv", xb, q, t["key"], t["value"], None, None, nh, nkv, hd, seq, pos)
    quantize(xq, xs, xb, d)
    if dtype == "f32":
        st.call("k_matmul_add", x, xb, w("wo"), d, d)
    else:
        st.call("k_matmul_q8_add", x, in_d, w("wo"), d, d, gs)
    st.call("k_rmsnorm", xb, x, t["norm_ffn"], d, EPS)
    quantize(xq, xs, xb, d)
    if dtype == "f32":
        st.call("k_matmul_swiglu", hb, xb, w("w1"), w("w3"), d, h)
        st.call("k_matmul_add", x, hb, w("w2"), h, d)
    else:
        st.call("k_matmul_q8_swiglu", hb, in_d, w("w1"), w("w3"), d, h, gs)
        quantize(hq, hs, hb, h)
        st.call("k_matmul_q8_add", x, in_h, w("w2"), h, d, gs)
    st.capture()
    st.out = {"x": x, "key": t["key"], "value": t["value"]}
    return st


def _vnni(w):
    """BF16 weights in the pack_bf16_vnni layout: 16-row tiles, K padded to 32, pairs of K side by side."""
    rows, cols = w.shape
    kp, rp = (cols + 31) // 32 * 32, (rows + 15) // 16 * 16
    p = torch.zeros(rp, kp, device="cuda", dtype=torch.bfloat16)
    p[:rows, :cols] = w
    return p.reshape(rp // 16, 16, kp // 2, 2).permute(0, 2, 1, 3).contiguous()


def _prepare_rows(c, seed):
    """The engine's batched calls of one layer, each call's rows the next one's input (layer) or rows given (prefill,
    batch); for sequences decoded together the calls are captured."""
    st = State()
    t, kv, seq = _inputs(c, seed)
    m, d, h, nh, nkv, gs, pos = c["rows"], c["dim"], c["hidden"], c["heads"], c["kv_heads"], c["gs"], c["pos"]
    hd, dtype = d // nh, c["dtype"]
    x, xb, q, k, v, hb = _empty(m, d), _empty(m, d), _empty(m, d), _empty(m, kv), _empty(m, kv), _empty(m, h)
    xq, xs = _empty(m, d, dtype=torch.int8), _empty(m, d // gs)
    hq, hs = _empty(m, h, dtype=torch.int8), _empty(m, h // gs)
    st.keep += [t, (x, xb, q, k, v, hb, xq, xs, hq, hs)]
    w = t
    if dtype == "bf16":
        w = {name: _vnni(t[name]) for name in _matrices(c)}
        st.keep.append(w)
        st.panel = lh.AlignedBuffer()
        st.lib.aligned_buffer_alloc(ctypes.byref(st.panel), st.lib.k_gemm_bf16_panel_bytes(m, max(d, h)), 1)

    def gemm(a, a_scales, cols, kind, *outs):
        """outs: (output, its columns, weight, W3 or None) of up to three matrices over the same rows."""
        if dtype == "q8":
            segs = (lh.GemmQ8Segment * len(outs))(*[
                lh.GemmQ8Segment(lh.ptr(o), n, lh.w8(*w[name]), lh.w8(*w[w3]) if w3 else lh.K8Weight(), None, None, n,
                                 kind) for o, n, name, w3 in outs])
            st.call("k_gemm_q8", a, a_scales, m, cols, gs, segs, len(outs))
        elif dtype == "bf16":
            segs = (lh.GemmBf16Segment * len(outs))(*[
                lh.GemmBf16Segment(lh.ptr(o), n, lh.ptr(w[name]), lh.ptr(w[w3]) if w3 else None, n, kind)
                for o, n, name, w3 in outs])
            st.call("k_gemm_bf16", a, cols, m, cols, segs, len(outs), ctypes.byref(st.panel))
        else:
            segs = (lh.GemmSegment * len(outs))(*[
                lh.GemmSegment(lh.ptr(o), n, lh.ptr(w[name]), lh.ptr(w[w3]) if w3 else None, cols, n, kind)
                for o, n, name, w3 in outs])
            st.call("k_gemm_f32", a, cols, m, cols, segs, len(outs))

    def norm(weight):
        if dtype == "q8":
            st.call("llhip_rmsnorm_quantize_rows", xq, xs, x, weight, m, d, EPS, gs)
        else:
            st.call("k_rmsnorm_rows", xb, x, weight, m, d, EPS)

    a, sa = (xq, xs) if dtype == "q8" else (xb, None)
    if dtype == "q8":
        st.call("k_embed_q8_rows", x, t["table"][0], t["table"][1], t["ids"], m, d, gs, TABLE_ROWS)
    else:
        st.call("k_embed_f32_rows", x, t["table"], t["ids"], m, d, TABLE_ROWS)
    norm(t["norm_att"])
    gemm(a, sa, d, lh.GEMM_STORE, (q, d, "wq", None), (k, kv, "wk", None), (v, kv, "wv", None))
    if c["kind"] == "batch":
        st.out = {"x": x, "h": hb, "q": q, "k": k, "v": v}
    else:
        st.call("llhip_rope_kv_store_rows", q, d, k, v, kv, t["rope"], 2 * hd, m, nh, nkv, hd, t["key"], t["value"], pos,
                seq)
        st.out = {"x": x, "key": t["key"], "value": t["value"]}
    if c["kind"] == "layer":
        _chained_rows(st, c, t, gemm, norm, seq, x, xb, q, hb, xq, xs, hq, hs)
        return st
    if c["kind"] == "prefill":
        st.call("k_attention_batch_kv", xb, q, t["key"], t["value"], None, None, nh, nkv, hd, seq, pos, m)
        st.out.update(h=hb, att=xb)

    def rows(src, cols, qq, ss):
        if dtype != "q8":
            return src, None
        st.call("k_quantize_rows", qq, ss, src, cols, m, cols, gs)
        return qq, ss

    gemm(*rows(t["att"], d, xq, xs), d, lh.GEMM_ADD, (x, d, "wo", None))
    gemm(*rows(t["mid"], d, xq, xs), d, lh.GEMM_SWIGLU, (hb, h, "w1", "w3"))
    gemm(*rows(t["gated"], h, hq, hs), h, lh.GEMM_ADD, (x, d, "w2", None))
    if c["kind"] == "batch":
        st.capture()
    return st


def _chained_rows(st, c, t, gemm, norm, seq, x, xb, q, hb, xq, xs, hq, hs):
    """The rest of a Q8_0 layer as the engine calls it, the rows quantized in the epilogues that the library has."""
    m, d, h, gs, hd = c["rows"], c["dim"], c["hidden"], c["gs"], c["dim"] // c["heads"]
    args = (c["heads"], c["kv_heads"], hd, seq, c["pos"], m)
    if hd % gs == 0:
        st.call("llhip_attention_batch_quantize", xq, xs, gs, xb, q, t["key"], t["value"], *args)
    else:
        st.call("k_attention_batch_kv", xb, q, t["key"], t["value"], None, None, *args)
        st.call("k_quantize_rows", xq, xs, xb, d, m, d, gs)
    gemm(xq, xs, d, lh.GEMM_ADD, (x, d, "wo", None))
    norm(t["norm_ffn"])
    w1, w3 = lh.w8(*t["w1"]), lh.w8(*t["w3"])
    segs = (lh.GemmQ8Segment * 1)(lh.GemmQ8Segment(lh.ptr(hb), h, w1, w3, None, None, h, lh.GEMM_SWIGLU))
    fused = (lh.ptr(xq), lh.ptr(xs), m, d, gs, ctypes.byref(w1), ctypes.byref(w3), h, lh.ptr(hq), lh.ptr(hs))
    plain = (lh.ptr(xq), lh.ptr(xs), m, d, gs, segs, 1)
    rows = (lh.ptr(hq), lh.ptr(hs), lh.ptr(hb), h, m, h, gs)
    lib = st.lib

    def swiglu():
        if not lib.llhip_gemm_q8_swiglu_quantize(*fused):
            lib.k_gemm_q8(*plain)
            lib.k_quantize_rows(*rows)

    st.calls.append((swiglu, ()))
    st.keep.append((w1, w3, segs))
    gemm(hq, hs, h, lh.GEMM_ADD, (x, d, "w2", None))


def _engine_inputs(c, seed):
    """The checkpoint's tensors (the classifier is the embedding) and the tokens."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))

    def weight(rows, cols, std):
        q, s = _quantize(torch.randn(rows, cols, generator=g, device="cuda") * std, c["gs"])
        return q.to(torch.int8), s.contiguous()

    # the embedding is the classifier too: its values stay small enough for logits of a few units
    t = {"embed": weight(VOCAB, c["dim"], 0.05)}
    for name, (rows, cols) in _matrices(c).items():
        t[name] = [weight(rows, cols, 0.02) for _ in range(c["layers"])]
    tokens = torch.randint(0, VOCAB, (c["rows"] + c["steps"],), generator=g, device="cuda").tolist()
    return t, tokens


def _context(c):
    return (c["rows"] + c["steps"] + 63) // 64 * 64


def _prepare_engine(c, seed):
    st = State()
    t, tokens = _engine_inputs(c, seed)
    cfg = {"dim": c["dim"], "hidden_dim": c["hidden"], "n_layers": c["layers"], "n_heads": c["heads"],
           "n_kv_heads": c["kv_heads"], "vocab_size": VOCAB, "seq_len": _context(c)}
    ones = np.ones((c["layers"], c["dim"]), np.float32)
    norms = {"rms_att": ones, "rms_ffn": ones, "rms_final": ones[0]}
    host = {"embed": tuple(a.cpu().numpy() for a in t["embed"])}
    for name in _matrices(c):
        host[name] = tuple([a[i].cpu().numpy() for a in t[name]] for i in range(2))
    del t
    fd, path = tempfile.mkstemp(suffix=".bin")
    os.close(fd)
    try:
        checkpoint.write_q8_v3(path, cfg, c["gs"], norms, host, shared=True)
        st.model = lh.Model()
        st.lib.engine_load_context(ctypes.byref(st.model), path.encode(), 0)
    finally:
        os.unlink(path)
    st.tokens, st.steps = (ctypes.c_int * len(tokens))(*tokens), c["steps"]
    return st


def run(state):
    if state.model is not None:
        return _run_engine(state)
    if state.graph:
        state.lib.llhip_graph_launch(state.graph)
    else:
        state.make()
    return state.out


def _run_engine(st):
    """The prompt's last logits, then each further token's, as the engine leaves them in host memory."""
    lib, model, vocab = st.lib, ctypes.byref(st.model), VOCAB
    total = len(st.tokens)
    rows = total - st.steps
    got = np.empty((st.steps + 1, vocab), np.float32)
    got[0] = np.ctypeslib.as_array(ctypes.cast(
        lib.engine_forward_batch(model, st.tokens, rows, 0, lh.LOGITS_LAST), ctypes.POINTER(ctypes.c_float)), (vocab,))
    for i in range(st.steps):
        got[1 + i] = np.ctypeslib.as_array(lib.engine_forward(model, st.tokens[rows + i], rows + i), (vocab,))
    return got


# ---- what a pass cannot do without -------------------------------------------------------------------------------


def _weight_bytes(c, count):
    if c["dtype"] in ("q8", "w8a32"):
        return count + 4 * count // c["gs"]
    return count * (2 if c["dtype"] == "bf16" else 4)


def work(case):
    c = case
    if c["kind"] == "gemv":
        count = c["n"] * c["d"]
        return {"bytes": _weight_bytes(c, count) + 4 * c["n"] + 4 * c["d"], "flops": 2 * count}
    layers = c.get("layers", 1)
    count = sum(r * k for r, k in _matrices(c).values()) * layers
    m, pos = c["rows"], c.get("pos", 0)
    kv = c["dim"] // c["heads"] * c["kv_heads"]
    reach = sum(range(pos + 1, pos + m + 1))  # (row, visible position) pairs
    if c["kind"] == "batch":
        return {"bytes": _weight_bytes(c, count) + 4 * m * (3 * c["dim"] + 2 * kv), "flops": 2 * m * count}
    total = {"bytes": _weight_bytes(c, count) + 8 * kv * (pos + m) * layers + 8 * m * c["dim"],
             "flops": 2 * m * count + 4 * c["dim"] * reach * layers}
    if c["kind"] == "engine":
        head, steps = VOCAB * c["dim"], c["steps"]
        total["bytes"] += steps * _weight_bytes(c, count) + (steps + 1) * (_weight_bytes(c, head) + 4 * VOCAB)
        total["bytes"] += sum(8 * kv * (m + i + 1) for i in range(steps)) * layers
        total["flops"] += 2 * steps * count + 2 * (steps + 1) * head
        total["flops"] += 4 * c["dim"] * layers * sum(m + i + 1 for i in range(steps))
    return total


def tolerance(case):
    """About four times the distance from exact() that the library showed over these ranges."""
    kind, dtype = case["kind"], case["dtype"]
    if kind in ("layer", "engine"):
        return {"rel": 0.03}  # ties along four or more chained quantizations: 0.0065 for a layer, 0.014 for two
    if kind == "decode" and dtype == "q8":
        return {"rel": 0.01}  # 2e-7 while no tie turns; one that does is followed by others, as in layer
    if kind in ("batch", "prefill") and dtype == "q8":
        return {"rel": 3e-4}  # 7e-5: ties of the first norm's rows alone; the sums themselves 2e-7
    if dtype == "bf16":
        return {"rel": 1e-4}  # 2e-5: likewise ties, of the rounding to BF16
    return {"rel": 6e-6 if kind == "prefill" else 2e-6}  # FP32 sums: 1.3e-6 over rows, 4e-7 in a decode token


# ---- the same in 64 bits -----------------------------------------------------------------------------------------


def _wide(w, gs):
    """A weight in float64, Q8_0 pairs multiplied out."""
    if not isinstance(w, tuple):
        return w.double()
    q, s = w
    return (q.double().reshape(q.shape[0], -1, gs) * s.double().reshape(q.shape[0], -1)[..., None]).reshape(q.shape)


def _rounded(x, c):
    """An activation as the products see it."""
    if c["dtype"] == "q8":
        q, s = _quantize(x, c["gs"])
        return (q.reshape(*s.shape, c["gs"]) * s[..., None]).reshape(x.shape)
    if c["dtype"] == "bf16":
        return x.float().bfloat16().double()
    return x


def _norm(x, w):
    return w * (x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS))


def _rotate(x, rope):
    """x: rows x heads x head_dim; rope: rows x 2 head_dim."""
    hd = x.shape[-1]
    swapped = x.reshape(*x.shape[:-1], hd // 2, 2).flip(-1).reshape(x.shape)
    return x * rope[:, None, :hd] + swapped * rope[:, None, hd:]


def _attend(q, key, value, pos):
    """q: rows x heads x head_dim; caches: KV heads x positions x head_dim; row i sees positions 0 .. pos + i."""
    m, nh, hd = q.shape
    nkv = key.shape[0]
    out = torch.empty_like(q)
    seen = torch.arange(pos + m, device=q.device)[None, :] <= torch.arange(pos, pos + m, device=q.device)[:, None]
    for h in range(nh):
        kh, vh = key[h // (nh // nkv), :pos + m], value[h // (nh // nkv), :pos + m]
        score = (q[:, h] @ kh.t().contiguous()) / np.sqrt(hd)
        out[:, h] = torch.softmax(score.masked_fill(~seen, float("-inf")), -1) @ vh
    return out


def _layer(c, t, x, key, value, pos, rope):
    """One decoder layer on float64 rows; the caches are written in place. Returns what the calls compute, by name."""
    m, nh, nkv, gs = x.shape[0], c["heads"], c["kv_heads"], c["gs"]
    hd = c["dim"] // nh

    def product(a, name):
        return _rounded(a, c) @ _wide(t[name], gs).t().contiguous()

    a = _norm(x, t["norm_att"].double())
    got = {"q": product(a, "wq"), "k": product(a, "wk"), "v": product(a, "wv")}
    if c["kind"] != "batch":
        q = _rotate(got["q"].reshape(m, nh, hd), rope)
        key[:, pos:pos + m] = _rotate(got["k"].reshape(m, nkv, hd), rope).transpose(0, 1)
        value[:, pos:pos + m] = got["v"].reshape(m, nkv, hd).transpose(0, 1)
        got.update(att=_attend(q, key, value, pos).reshape(m, -1), key=key, value=value)
    x = x + product(t["att"].double() if "att" in t else got["att"], "wo")
    b = t["mid"].double() if "mid" in t else _norm(x, t["norm_ffn"].double())
    gate = product(b, "w1")
    got["h"] = gate / (1.0 + torch.exp(-gate)) * product(b, "w3")
    got["x"] = x + product(t["gated"].double() if "gated" in t else got["h"], "w2")
    return got


def exact(case, seed):
    c = case
    if c["kind"] == "gemv":
        x, wq, ws = _gemv_inputs(c, seed)
        return _rounded(x.double()[None], c)[0] @ _wide((wq, ws), c["gs"]).t().contiguous()
    if c["kind"] == "engine":
        return _exact_engine(c, seed)
    t, _, _ = _inputs(c, seed)
    x = _wide(t["table"], c["gs"])[t["ids"].long()]
    key, value = t["key"].double(), t["value"].double()
    got = _layer(c, t, x, key, value, c["pos"], t["rope"].double())
    if c["kind"] == "decode":
        got["x"] = got["x"][0]
    if c["kind"] == "layer":
        got["x"] = None  # a chain of quantized rows: which way its ties fall is not the precision of any one product
    names = {"batch": ("x", "h", "q", "k", "v"), "prefill": ("x", "h", "att", "key", "value")}
    return {name: got[name] for name in names.get(c["kind"], ("x", "key", "value"))}


def _exact_engine(c, seed):
    t, tokens = _engine_inputs(c, seed)
    hd, m = c["dim"] // c["heads"], c["rows"]
    # the engine rotates by float32 tables of float32 angles
    f = np.float32
    freq = (f(1.0) / np.power(f(500000.0), (np.arange(0, hd, 2).astype(f) / f(hd)).astype(f))).astype(f)
    angle = (np.arange(len(tokens)).astype(f)[:, None] * freq).astype(f)
    cos, sin = np.repeat(np.cos(angle), 2, 1), np.stack((-np.sin(angle), np.sin(angle)), -1).reshape(len(tokens), hd)
    rope = torch.from_numpy(np.concatenate((cos, sin), 1)).cuda().double()
    embed = _wide(t["embed"], c["gs"])
    ones = torch.ones(c["dim"], device="cuda", dtype=torch.float64)
    caches = [torch.zeros(2, c["kv_heads"], len(tokens), hd, device="cuda", dtype=torch.float64)
              for _ in range(c["layers"])]
    got = []
    for first, count in [(0, m)] + [(m + i, 1) for i in range(c["steps"])]:
        x = embed[torch.tensor(tokens[first:first + count], device="cuda")]
        for l, cache in enumerate(caches):
            layer = {name: t[name][l] for name in _matrices(c)}
            layer.update(norm_att=ones, norm_ffn=ones)
            x = _layer(c, layer, x, cache[0], cache[1], first, rope[first:first + count])["x"]
        got.append(_rounded(_norm(x[-1:], ones), c)[0] @ embed.t().contiguous())
    return torch.stack(got)
