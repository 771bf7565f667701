"""Workloads whose speed this framework is judged by, each through its public entry points.

Five kinds of work, over the layer shapes of Gemma-4-E2B (`E2BShape()`, the uniform layer, and `E2BShape.real()`, the
model's own layout with head dim 512 globals, FFN 12288, shared K/V caches and per-layer embeddings):

* "matvec":  one quantized matrix times one vector;
* "head":    final norm, LM head, softcap and sampling for a batch of vectors;
* "decode":  one token of one sequence (`Decoder`, the captured step);
* "batch":   one token for each of many ragged sequences (`BatchDecoder`, the captured step);
* "prefill": a prompt (`BatchDecoder.prefill`), from position 0 or after earlier turns.

`layers` below 35 takes a slice of the model without its LM head and returns the residual stream; 35 is the whole call
and returns logits. Weights are random blocks of the file formats with the spread of a trained model (zero mean, 6-bit
scales in use), so that no layer's GELU saturates and no softmax is one-hot. Everything is made from the seed by torch;
`exact` computes the same in float64 from the same tensors.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gemma4-webgpu_amd"))

from g4hip import Context  # noqa: E402
from g4hip.decoder import BatchDecoder, Decoder, E2BShape  # noqa: E402
from g4hip.device import Buffer  # noqa: E402

DEV = "cuda"
VOCAB = 262144
HIDDEN = 1536
PAGE = 16
F64 = torch.float64


def listed():
    return [
        # the smallest call a per-kernel host makes: the FFN gate matrix times one vector
        {"name": "matvec-6144x1536", "kind": "matvec", "rows": 6144, "width": 1536, "wtype": "q4k"},
        # sampling for a handful of sequences: the LM head at 8 vectors, top-k candidates for a host sampler
        {"name": "head-8", "kind": "head", "vectors": 8, "wtype": "q6k", "sample": "topk"},
        # a slice of the single-stream step (four window layers, one global) at a short chat's context
        {"name": "layers-1", "kind": "decode", "layout": "uniform", "layers": 5, "position": 512},
        # the same at a long document's context on the model's own layout (head dim 512 globals, shared caches)
        {"name": "layers-1-long", "kind": "decode", "layout": "real", "layers": 10, "position": 32000},
        # a slice of a lightly loaded server's step: few sequences of mixed length
        {"name": "layers-7", "kind": "batch", "layout": "uniform", "layers": 5, "sequences": 7, "longest": 8192},
        # a slice of a full server's step on the model's own layout
        {"name": "layers-64", "kind": "batch", "layout": "real", "layers": 10, "sequences": 64, "longest": 4096},
        # interactive chat: one token of one sequence, whole model
        {"name": "decode-1", "kind": "decode", "layout": "uniform", "layers": 35, "position": 512},
        # the same on the model's own layout, some turns into the chat
        {"name": "decode-1-real", "kind": "decode", "layout": "real", "layers": 35, "position": 1777},
        # a server's step over 32 ragged sequences, whole model
        {"name": "decode-32", "kind": "batch", "layout": "uniform", "layers": 35, "sequences": 32, "longest": 8192},
        # a short user turn after an earlier conversation
        {"name": "prefill-27", "kind": "prefill", "layout": "real", "layers": 35, "tokens": 27, "start": 700,
         "rows": 64},
        # a page of prompt
        {"name": "prefill-512", "kind": "prefill", "layout": "uniform", "layers": 35, "tokens": 512, "start": 0,
         "rows": 64},
        # a prompt that nearly fills the default 2048-token context
        {"name": "prefill-1900", "kind": "prefill", "layout": "real", "layers": 35, "tokens": 1900, "start": 0,
         "rows": 64},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("matvec", "head", "decode", "batch", "batch", "prefill", "prefill", "prefill"))
    layout = rng.choice(("uniform", "real"))
    layers = rng.choice((5, 15)) if layout == "uniform" else rng.choice((10, 20))
    if kind == "matvec":
        wtype = rng.choice(("q4k", "q6k"))
        width = rng.choice((1536, 2048, 4096, 6144, 12288))
        return {"kind": kind, "rows": _log_int(rng, 256, 16384), "width": width, "wtype": wtype}
    if kind == "head":
        return {"kind": kind, "vectors": _log_int(rng, 1, 64), "wtype": rng.choice(("q6k", "q6k", "q4k", "f16")),
                "sample": rng.choice(("argmax", "topk"))}
    if kind == "decode":
        return {"kind": kind, "layout": layout, "layers": layers, "position": _log_int(rng, 16, 32700)}
    if kind == "batch":
        return {"kind": kind, "layout": layout, "layers": layers, "sequences": _log_int(rng, 2, 64),
                "longest": _log_int(rng, 256, 8192)}
    start = rng.choice((0, 0, _log_int(rng, 16, 2000)))
    return {"kind": kind, "layout": layout, "layers": layers, "tokens": _log_int(rng, 8, 1900), "start": start,
            "rows": rng.choice((16, 32, 64, 64))}


# ---- inputs, from the seed alone ------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _bytes(g, *shape):
    """Random bytes, drawn eight at a time."""
    n = math.prod(shape)
    w = torch.randint(-2 ** 63, 2 ** 63 - 1, (-(-n // 8),), dtype=torch.int64, device=DEV, generator=g)
    return w.view(torch.uint8)[:n].view(*shape)


def _scales(g, nb, lo=24):
    """Eight 6-bit scales per block and mins near them (zero-mean sub-blocks), and the 12 bytes that pack both."""
    r = _bytes(g, nb, 16).int()
    sc = lo + r[:, :8] % (64 - lo)
    mn = (sc + r[:, 8:] % 7 - 3).clamp(0, 63)
    packed = torch.cat([(sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6), (mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6),
                        (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1).to(torch.uint8)
    return sc, mn, packed


def _d(g, nb, value):
    return (value * (0.8 + 0.4 * torch.rand(nb, 1, device=DEV, generator=g))).half()


def _q4k(g, rows, width, std=0.03):
    """Q4_K blocks [rows * width / 256][144]: nibbles uniform, scale times 7.5 taken off by the min."""
    nb = rows * width // 256
    d = _d(g, nb, std / (44 * 4.6))
    dmin = (d.float() * 7.5).half()
    _, _, packed = _scales(g, nb)
    return torch.cat([d.view(torch.uint8), dmin.view(torch.uint8), packed, _bytes(g, nb, 128)], 1)


def _q5k(g, nb, std=0.05):
    """Q5_K blocks [nb][176] (the per-layer embedding table)."""
    d = _d(g, nb, std / (44 * 9.2))
    dmin = (d.float() * 15.5).half()
    _, _, packed = _scales(g, nb)
    return torch.cat([d.view(torch.uint8), dmin.view(torch.uint8), packed, _bytes(g, nb, 160)], 1)


def _q6k(g, rows, width, std=0.03):
    """Q6_K blocks [rows * width / 256][210]: signed 8-bit scales of 32 .. 127, codes uniform."""
    nb = rows * width // 256
    r = _bytes(g, nb, 16).int()
    sc = ((32 + (r & 127) * 95 // 127) * (1 - 2 * (r >> 7))).to(torch.int8)
    return torch.cat([_bytes(g, nb, 192), sc.view(torch.uint8), _d(g, nb, std / (84 * 18.5)).view(torch.uint8)], 1)


def _half(g, n, mean, std):
    return (mean + std * torch.randn(n, device=DEV, generator=g)).half()


def _normal(g, *shape):
    return torch.randn(*shape, device=DEV, generator=g)


MATRICES = {"q4k": _q4k, "q6k": _q6k, "f16": lambda g, rows, width: _half(g, rows * width, 0.0, 0.03)}


def _shape(case):
    layers = case["layers"]
    if case["layout"] == "uniform":
        return E2BShape(n_layers=layers)
    # the slice keeps the model's order: layers with caches of their own first, then layers that share them
    return E2BShape.real(n_layers=layers, n_unshared=15 if layers == 35 else layers // 2)


def _layer(s, il, g):
    """The tensors of layer il, as a file would hold them."""
    h, q, kv, f, hd = s.hidden, s.q_dim_of(il), s.kv_dim_of(il), s.ffn_of(il), s.hd(il)
    own = s.is_producer(il)
    w = {"wq": _q4k(g, q, h), "wk": _q4k(g, kv, h) if own else None, "wv": _q4k(g, kv, h) if own else None,
         "wo": _q4k(g, h, q), "wgate": _q4k(g, f, h), "wup": _q4k(g, f, h), "wdown": _q6k(g, h, f),
         "q_norm": _half(g, hd, 0.3, 0.03), "k_norm": _half(g, hd, 0.3, 0.03) if own else None}
    for name in ("attn_norm", "pre_ffn_norm"):
        w[name] = _half(g, h, 1.0, 0.1)
    for name in ("post_attn_norm", "post_ffn_norm"):  # each layer adds a part of the residual stream's size
        w[name] = _half(g, h, 0.25, 0.03)
    if s.ple_dim:
        w["ple_gate"] = _half(g, s.ple_dim * h, 0.0, 0.03)
        w["ple_proj"] = _half(g, h * s.ple_dim, 0.0, 0.03)
        w["ple_post_norm"] = _half(g, h, 0.25, 0.03)
        w["ple_scale"] = _half(g, 2, 0.98, 0.01)
    return w


def _globals(s, g, head):
    """The tensors outside the layers."""
    w = {"embedding": _half(g, s.vocab * s.hidden, 0.0, 0.03), "final_norm": _half(g, s.hidden, 1.0, 0.1)}
    if head:
        w["lm_head"] = _q6k(g, s.vocab, s.hidden)
    if s.ple_dim:
        w["ple_model_proj"] = _half(g, s.n_layers * s.ple_dim * s.hidden, 0.0, 0.03)
        w["ple_proj_norm"] = _half(g, s.ple_dim, 1.0, 0.1)
        w["ple_table"] = _q5k(g, s.vocab * s.n_layers)
    return w


def _cached(s, il, rows, g):
    """Cached K and V rows of layer il: normalised vectors, K under its norm weight."""
    n = rows * s.kv_dim_of(il)
    return _half(g, n, 0.0, 0.3).view(rows, -1), _half(g, n, 0.0, 1.0).view(rows, -1)


def _lengths(case, seed):
    """Cached lengths before the step: spread evenly over 128 .. longest, in an order of the seed's."""
    low = min(128, case["longest"] // 2)
    lens = np.linspace(low, case["longest"] - 1, case["sequences"]).astype(np.int64)
    return np.random.default_rng(seed).permutation(lens)


def _tokens(seed, n):
    return np.random.default_rng(seed + 1).integers(0, VOCAB, n).astype(np.uint32)


def _page_order(seed, pages):
    """Where a serving loop's page list has scattered a sequence's pages."""
    return np.random.default_rng(seed + 2).permutation(pages).astype(np.int32)


# ---- states ---------------------------------------------------------------------------------------------------------

_context = None


def _ctx():
    global _context
    if _context is None:
        _context = Context(0)
    return _context


class _Graph:
    """A captured sequence of launches, destroyed with the state that holds it."""

    def __init__(self, ctx, enqueue):
        self.ctx = ctx
        ctx.graph_begin()
        try:
            enqueue()
        finally:
            self.graph = ctx.graph_end()

    def launch(self):
        self.ctx.graph_launch(self.graph)

    def __del__(self):
        self.ctx.graph_destroy(self.graph)


def _on(ctx, t):
    """A torch tensor's memory as a buffer of the framework."""
    return Buffer(ctx, t.data_ptr(), t.numel() * t.element_size(), owned=False)


def _put(ctx, buf, t):
    ctx.copy(buf, t.data_ptr(), t.numel() * t.element_size())


def _fill_model(ctx, d, seed, head, rows):
    """Gives a decoder its weights and its cached rows; returns the cache tensors the decoder now uses."""
    s, caches = d.s, {}
    for il, layer in enumerate(d.layers):
        g = _gen(seed * 1009 + il)
        w = _layer(s, il, g)
        if s.is_producer(il):
            caches[il] = _cached(s, il, rows, g)
        torch.cuda.synchronize()
        for name, t in w.items():
            if t is not None:
                _put(ctx, getattr(layer, name), t)
        ctx.sync()
        layer.k_cache, layer.v_cache = (_on(ctx, t) for t in caches[s.producer(il)])
    w = _globals(s, _gen(seed * 1009 + 999), head)
    torch.cuda.synchronize()
    for name, t in w.items():
        _put(ctx, getattr(d, name), t)
    ctx.sync()
    return caches


def _last_caches(s, caches):
    """The caches of the deepest window layer and the deepest global layer that have their own."""
    last = {s.is_global(il): il for il in sorted(caches)}
    return [t for il in sorted(last.values()) for t in caches[il]]


def _prepare_decode(case, seed):
    ctx, s, pos = _ctx(), _shape(case), case["position"]
    head = case["layers"] == 35
    max_seq = -(-(pos + 64) // PAGE) * PAGE
    d = Decoder(ctx, s, max_seq=max_seq, seed=1, lm_head=head, embed=True)
    caches = _fill_model(ctx, d, seed, head, max_seq)
    out = torch.zeros(VOCAB if head else HIDDEN, device=DEV)
    setattr(d, "logits" if head else "hidden", _on(ctx, out))
    torch.cuda.synchronize()
    # the token and the position the host hands each step (it samples by its own rules)
    token = ctx.from_numpy(_tokens(seed, 1))
    position = ctx.from_numpy(np.array([pos], np.uint32))
    ctx.copy(d.token, token, 4)
    ctx.copy(d.pos, position, 4)
    graph = _Graph(ctx, d.step_fused)
    ctx.sync()
    return {"kind": "decode", "ctx": ctx, "decoder": d, "token": token, "position": position, "graph": graph,
            "keep": caches, "out": [out] + _last_caches(s, caches)}


def _prepare_batch(case, seed):
    ctx, s, n = _ctx(), _shape(case), case["sequences"]
    head = case["layers"] == 35
    lens = _lengths(case, seed)
    d = BatchDecoder(ctx, lens, s, reserve=PAGE, seed=1, lm_head=head, embed=True)
    table = _batch_table(lens, seed)
    d.page_table.upload(np.pad(table, ((0, 0), (0, d.max_pages - table.shape[1])), constant_values=-1))
    caches = _fill_model(ctx, d, seed, head, d.num_pages * PAGE)
    out = torch.zeros(n, VOCAB if head else HIDDEN, device=DEV)
    setattr(d, "logits" if head else "hidden", _on(ctx, out))
    torch.cuda.synchronize()
    tokens = ctx.from_numpy(_tokens(seed, n))
    lengths = ctx.from_numpy(lens.astype(np.uint32))
    ctx.copy(d.tokens, tokens, 4 * n)
    ctx.copy(d.seq_lens, lengths, 4 * n)
    graph = _Graph(ctx, d.step)
    ctx.sync()
    return {"kind": "batch", "ctx": ctx, "decoder": d, "tokens": tokens, "lengths": lengths, "graph": graph,
            "keep": caches, "out": [out] + _last_caches(s, caches)}


def _batch_table(lens, seed):
    """Page lists of ragged sequences (16 rows reserved for each), scattered over the pool."""
    per = [-(-(int(n) + PAGE) // PAGE) for n in lens]
    order = _page_order(seed, sum(per))
    table, at = np.full((len(per), max(per)), -1, np.int32), 0
    for i, n in enumerate(per):
        table[i, :n] = order[at:at + n]
        at += n
    return table


def _prefill_pages(case):
    return -(-(case["start"] + case["tokens"] + PAGE) // PAGE)


def _prepare_prefill(case, seed):
    ctx, s = _ctx(), _shape(case)
    head = case["layers"] == 35
    d = BatchDecoder(ctx, [0] * case["rows"], s, reserve=_prefill_pages(case) * PAGE, seed=1, lm_head=head,
                     shared_pages=True, embed=True)
    order = _page_order(seed, d.num_pages)
    d.page_table_host = np.repeat(order[None, :], d.B, 0)
    d.page_table.upload(d.page_table_host)
    caches = _fill_model(ctx, d, seed, head, d.num_pages * PAGE)
    out = torch.zeros(case["rows"], VOCAB if head else HIDDEN, device=DEV)
    setattr(d, "logits" if head else "hidden", _on(ctx, out))
    torch.cuda.synchronize()
    return {"kind": "prefill", "ctx": ctx, "decoder": d, "prompt": _tokens(seed, case["tokens"]),
            "start": case["start"], "keep": caches, "out": out, "caches": _last_caches(s, caches)}


def _head_tensors(case, seed):
    g = _gen(seed)
    return (MATRICES[case["wtype"]](g, VOCAB, HIDDEN), _half(g, HIDDEN, 1.0, 0.1),
            _normal(g, case["vectors"], HIDDEN))


def _prepare_head(case, seed):
    ctx, n, wtype = _ctx(), case["vectors"], case["wtype"]
    w, norm, x = _head_tensors(case, seed)
    top = case["sample"] == "topk"
    logits = torch.zeros(n, VOCAB, device=DEV)
    pairs = torch.zeros(n, 512, device=DEV)
    tokens = torch.zeros(n, dtype=torch.int32, device=DEV)
    xn = torch.zeros(n, HIDDEN, device=DEV)
    ops = ctx.alloc(ctx.batch_operand_bytes(HIDDEN, n))
    torch.cuda.synchronize()
    p = torch.Tensor.data_ptr

    def enqueue():
        if n == 1 and wtype != "f16":
            if top:
                ctx.normAddMatmulTopk(wtype, p(x), p(norm), None, None, None, p(w), p(logits), VOCAB, HIDDEN, p(pairs),
                                      softcap=30.0)
            else:
                ctx.normAddMatmulArgmax(wtype, p(x), p(norm), None, None, None, p(w), p(logits), VOCAB, HIDDEN,
                                        p(tokens), softcap=30.0)
            return
        ctx.batchPrep(p(x), 1, p(norm), None, None, None, p(xn), HIDDEN, n, ops=ops)
        if wtype == "f16":
            ctx.matmulF16(p(xn), p(w), p(logits), VOCAB, HIDDEN, n)
            ctx.logitSoftcap(p(logits), n * VOCAB, 30.0)
        else:
            ctx.matmulSegmentsBatchPartial(wtype, p(xn), [p(w)], [p(logits)], [VOCAB], HIDDEN, n, 1, ops=ops,
                                           softcap=30.0)
        if top:
            ctx.topk256Batch(p(logits), p(pairs), VOCAB, n)
        else:
            ctx.argmaxBatch(p(logits), p(tokens), VOCAB, n)

    graph = _Graph(ctx, enqueue)
    ctx.sync()
    return {"kind": "head", "graph": graph, "keep": (w, norm, x, xn, ops, tokens),
            "out": [logits, pairs] if top else [logits]}


def _prepare_matvec(case, seed):
    g = _gen(seed)
    w = MATRICES[case["wtype"]](g, case["rows"], case["width"])
    x = _normal(g, case["width"])
    y = torch.zeros(case["rows"], device=DEV)
    torch.cuda.synchronize()
    return {"kind": "matvec", "ctx": _ctx(), "case": case, "w": w, "x": x, "out": y}


def prepare(case, seed):
    return {"matvec": _prepare_matvec, "head": _prepare_head, "decode": _prepare_decode, "batch": _prepare_batch,
            "prefill": _prepare_prefill}[case["kind"]](case, seed)


def run(state):
    kind = state["kind"]
    if kind == "matvec":
        c = state["case"]
        state["ctx"].matmulQuant(state["x"].data_ptr(), state["w"].data_ptr(), state["out"].data_ptr(), c["rows"],
                                 c["width"], c["wtype"])
        return state["out"]
    if kind == "head":
        state["graph"].launch()
        return state["out"]
    ctx, d = state["ctx"], state["decoder"]
    if kind == "decode":
        ctx.copy(d.token, state["token"], 4)
        ctx.copy(d.pos, state["position"], 4)
        state["graph"].launch()
        return state["out"]
    if kind == "batch":
        ctx.copy(d.tokens, state["tokens"], 4 * d.B)
        ctx.copy(d.seq_lens, state["lengths"], 4 * d.B)
        state["graph"].launch()
        return state["out"]
    row = d.prefill(state["prompt"], state["start"])
    return [state["out"][row]] + state["caches"]


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

def _matrix_bytes(rows, width, wtype):
    return rows * width * {"q4k": 144 / 256, "q6k": 210 / 256, "f16": 2.0}[wtype]


def work(case):
    kind = case["kind"]
    if kind == "matvec":
        m, n = case["rows"], case["width"]
        return {"bytes": _matrix_bytes(m, n, case["wtype"]) + 4 * (m + n), "flops": 2.0 * m * n}
    if kind == "head":
        n = case["vectors"]
        return {"bytes": _matrix_bytes(VOCAB, HIDDEN, case["wtype"]) + 4.0 * n * (HIDDEN + VOCAB),
                "flops": 2.0 * n * VOCAB * HIDDEN}
    s = _shape(case)
    head = case["layers"] == 35
    if kind == "decode":
        rows, last, ends = 1, 1, [case["position"] + 1]
    elif kind == "batch":
        rows = last = case["sequences"]
        ends = [int(n) + 1 for n in _lengths(case, 0)]
    else:
        rows, last, ends = case["tokens"], 1, [case["start"] + t + 1 for t in range(case["tokens"])]
    # weights, embedding rows and per-layer embeddings once; the head for the sampled rows only
    weights = s.weight_bytes() + (s.lm_head_bytes() if head else 0)
    out_row = 4 * VOCAB if head else 4 * HIDDEN
    nbytes = weights + rows * 2 * HIDDEN + last * out_row
    flops = 2.0 * (last * VOCAB * HIDDEN if head else 0)
    if s.ple_dim:
        nbytes += s.n_layers * (3 * s.ple_dim * HIDDEN * 2 + rows * 176)
        flops += 2.0 * rows * s.n_layers * 3 * s.ple_dim * HIDDEN
    for il in range(s.n_layers):
        q, kv, own = s.q_dim_of(il), s.kv_dim_of(il), s.is_producer(il)
        flops += 2.0 * rows * HIDDEN * (2 * q + (2 * kv if own else 0) + 3 * s.ffn_of(il))
        spans = [e if s.is_global(il) else min(e, s.window) for e in ends]
        flops += 4.0 * sum(spans) * q
        if kind == "prefill":  # one sequence: its cached rows once, the new ones written and read
            first = 0 if s.is_global(il) else max(0, case["start"] - s.window)
            nbytes += 4 * kv * (case["start"] - first) + (4 * kv * rows if own else 0)
        else:
            nbytes += 4 * kv * sum(spans)
    return {"bytes": float(nbytes), "flops": flops}


# ---- the same in float64 --------------------------------------------------------------------------------------------

def _q4k_values(b, rows, width):
    b = b.view(-1, 144)
    d, dmin = (b[:, i:i + 2].contiguous().view(torch.float16).to(F64) for i in (0, 2))
    sc, mn = _unpack_scales(b[:, 4:16])
    q = b[:, 16:].reshape(-1, 4, 1, 32)
    code = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).to(F64)
    return ((d * sc)[:, :, None] * code - (dmin * mn)[:, :, None]).view(rows, width)


def _unpack_scales(p):
    p = p.int()
    lo, mid, hi = p[:, :4], p[:, 4:8], p[:, 8:]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1)
    mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1)
    return sc.to(F64), mn.to(F64)


def _q5k_values(b):
    b = b.view(-1, 176)
    d, dmin = (b[:, i:i + 2].contiguous().view(torch.float16).to(F64) for i in (0, 2))
    sc, mn = _unpack_scales(b[:, 4:16])
    q = b[:, 48:].reshape(-1, 4, 1, 32)
    code = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).int()
    high = (b[:, 16:48].int()[:, None, :] >> torch.arange(8, device=DEV)[None, :, None]) & 1
    return ((d * sc)[:, :, None] * (code + 16 * high).to(F64) - (dmin * mn)[:, :, None]).view(-1, 256)


def _q6k_values(b, rows, width):
    b = b.view(-1, 210)
    ql, qh = b[:, :128].reshape(-1, 2, 64), b[:, 128:192].reshape(-1, 2, 32)
    lo = torch.cat([ql[..., :32] & 15, ql[..., 32:] & 15, ql[..., :32] >> 4, ql[..., 32:] >> 4], 2)
    hi = torch.cat([(qh >> i) & 3 for i in (0, 2, 4, 6)], 2)
    code = (lo | (hi << 4)).reshape(-1, 16, 16).to(F64) - 32
    sc = b[:, 192:208].contiguous().view(torch.int8).to(F64)
    d = b[:, 208:210].contiguous().view(torch.float16).to(F64)
    return ((d * sc)[:, :, None] * code).view(rows, width)


def _times(x, w, rows, wtype):
    """x [n][width] times a matrix of the file's format, in float64, a slice of rows at a time."""
    width, out = x.shape[-1], []
    values = {"q4k": _q4k_values, "q6k": _q6k_values, "f16": lambda t, r, c: t.to(F64).view(r, c)}[wtype]
    per = w.numel() // rows
    for r in range(0, rows, 32768):
        n = min(32768, rows - r)
        out.append(x @ values(w.view(-1)[r * per:(r + n) * per], n, width).T)
    return torch.cat(out, 1)


def _rms(x, w=None):
    y = x / torch.sqrt(x.square().mean(-1, keepdim=True) + 1e-6)
    return y if w is None else y * w.to(F64)


def _gelu(x):
    t = (0.7978845608028654 * x * (1 + 0.044715 * x * x)).clamp(-15, 15)
    return 0.5 * x * (1 + torch.tanh(t))


def _rope(x, positions, glob, s):
    """Rotate-half over x [n][heads][dim]; the angle is the float32 product of position and frequency."""
    dim = x.shape[-1]
    half = dim // 2
    i = torch.arange(half, device=DEV, dtype=F64)
    freq = (1 / torch.tensor(s.theta_global if glob else s.theta_local, dtype=F64, device=DEV) ** (2 * i / dim)).float()
    if glob:  # the proportional table rotates a quarter of the pairs
        freq = torch.where(i < half // 4, freq, torch.zeros_like(freq))
    a = (positions.float()[:, None] * freq[None, :]).to(F64)[:, None, :]
    c, sn = torch.cos(a), torch.sin(a)
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat([lo * c - hi * sn, lo * sn + hi * c], -1)


def _attend(q, k, v, positions, window, sequences):
    """q [n][heads][dim] over pool rows; `sequences` gives each sequence's queries and its pool rows by position."""
    out = torch.empty_like(q)
    for rows, at in sequences:
        pos = positions[rows]
        end = int(pos.max()) + 1
        first = max(0, int(pos.min()) + 1 - window) if window else 0
        kk, vv = k[at[first:end]].to(F64), v[at[first:end]].to(F64)
        t = torch.arange(first, end, device=DEV)
        dead = t[None, :] > pos[:, None]
        if window:
            dead |= t[None, :] <= pos[:, None] - window
        for r in range(0, len(rows), 256):
            m = rows[r:r + 256]
            sc = (q[m] @ kk.T).masked_fill(dead[r:r + 256, None, :], -math.inf)
            out[m] = torch.softmax(sc, -1) @ vv
    return out


def _exact_model(case, seed, tokens, positions, rows, sequences):
    s = _shape(case)
    head = case["layers"] == 35
    w = _globals(s, _gen(seed * 1009 + 999), head)
    n = len(tokens)
    at = torch.from_numpy(tokens.astype(np.int64)).to(DEV)
    x = w["embedding"].view(-1, HIDDEN)[at].to(F64) * math.sqrt(HIDDEN)
    D, L = s.ple_dim, s.n_layers
    if D:
        p = _rms(_times(x, w["ple_model_proj"], L * D, "f16").view(n, L, D), w["ple_proj_norm"])
        t = _q5k_values(w["ple_table"].view(-1, L * 176)[at].contiguous()).half().to(F64).view(n, L, D)
        ple = (p + t * math.sqrt(D)) / math.sqrt(2)
    pools = {}
    where = torch.empty(n, dtype=torch.int64, device=DEV)
    for queries, slot in sequences:
        where[queries] = slot[positions[queries]]
    for il in range(L):
        g = _gen(seed * 1009 + il)
        lw = _layer(s, il, g)
        qd, kvd, f, hd, glob = s.q_dim_of(il), s.kv_dim_of(il), s.ffn_of(il), s.hd(il), s.is_global(il)
        src = s.producer(il)
        xn = _rms(x, lw["attn_norm"])
        q = _rope(_rms(_times(xn, lw["wq"], qd, "q4k").view(n, s.n_q_heads, hd), lw["q_norm"]), positions, glob, s)
        if src == il:
            k = _rope(_rms(_times(xn, lw["wk"], kvd, "q4k").view(n, 1, hd), lw["k_norm"]), positions, glob, s)
            v = _rms(_times(xn, lw["wv"], kvd, "q4k").view(n, 1, hd))
            pools[il] = _cached(s, il, rows, g)
            for pool, row in zip(pools[il], (k, v)):
                pool[where] = row.view(n, kvd).half()
        a = _attend(q, *pools[src], positions, 0 if glob else s.window, sequences).view(n, qd)
        h = x + _rms(_times(a, lw["wo"], HIDDEN, "q4k"), lw["post_attn_norm"])
        hn = _rms(h, lw["pre_ffn_norm"])
        act = _gelu(_times(hn, lw["wgate"], f, "q4k")) * _times(hn, lw["wup"], f, "q4k")
        x = h + _rms(_times(act, lw["wdown"], HIDDEN, "q6k"), lw["post_ffn_norm"])
        if D:
            t = _gelu(_times(x, lw["ple_gate"], D, "f16")) * ple[:, il]
            x = (x + _rms(_times(t, lw["ple_proj"], HIDDEN, "f16"), lw["ple_post_norm"])) * lw["ple_scale"][0].to(F64)
    caches = _last_caches(s, pools)
    if case["kind"] == "prefill":
        x = x[-1:]
    if head:
        x = 30 * torch.tanh(_times(_rms(x, w["final_norm"]), w["lm_head"], VOCAB, "q6k") / 30)
    return [x if case["kind"] == "batch" else x[0]] + caches


def exact(case, seed):
    kind = case["kind"]
    if kind == "matvec":
        g = _gen(seed)
        w = MATRICES[case["wtype"]](g, case["rows"], case["width"])
        return _times(_normal(g, case["width"])[None].to(F64), w, case["rows"], case["wtype"])[0]
    if kind == "head":
        w, norm, x = _head_tensors(case, seed)
        logits = 30 * torch.tanh(_times(_rms(x.to(F64), norm), w, VOCAB, case["wtype"]) / 30)
        if case["sample"] != "topk":
            return [logits]
        best = logits.view(case["vectors"], -1, 256).max(1)
        index = (best.indices * 256 + torch.arange(256, device=DEV)).int().view(torch.float32)
        return [logits, torch.stack([best.values, index.to(F64)], 2).view(case["vectors"], 512)]
    if kind == "decode":
        rows = -(-(case["position"] + 64) // PAGE) * PAGE
        return _exact_model(case, seed, _tokens(seed, 1), torch.tensor([case["position"]], device=DEV), rows,
                            [(torch.tensor([0], device=DEV), torch.arange(rows, device=DEV))])
    slot = torch.arange(PAGE, device=DEV)
    if kind == "batch":
        lens = _lengths(case, seed)
        table = _batch_table(lens, seed)
        sequences = [(torch.tensor([i], device=DEV),
                      (torch.from_numpy(table[i]).to(DEV).long()[:, None] * PAGE + slot).view(-1))
                     for i in range(len(lens))]
        rows = int(sum(-(-(int(n) + PAGE) // PAGE) for n in lens)) * PAGE
        return _exact_model(case, seed, _tokens(seed, len(lens)), torch.from_numpy(lens).to(DEV), rows, sequences)
    pages = _prefill_pages(case)
    at = (torch.from_numpy(_page_order(seed, pages)).to(DEV).long()[:, None] * PAGE + slot).view(-1)
    n = case["tokens"]
    return _exact_model(case, seed, _tokens(seed, n), case["start"] + torch.arange(n, device=DEV), pages * PAGE,
                        [(torch.arange(n, device=DEV), at)])


# About four times what the paths differ by from float64: 4e-5 where activations become 16-bit fixed point per 32 values
# (one vector), 1.4e-4 where a Q6_K weight's scale times code rounds once to f16 (many vectors), and what a stack of
# layers makes of these (1.5e-4 for one vector, 4e-4 with the f16 rows a prompt appends).
TOLERANCE = {"matvec": 2e-4, "head": 6e-4, "decode": 8e-4, "batch": 1.5e-3, "prefill": 2e-3}


def tolerance(case):
    return {"rel": TOLERANCE[case["kind"]]}
