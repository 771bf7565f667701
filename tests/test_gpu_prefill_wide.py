"""GPU parity of the whole-prompt path: the prefill matmuls against a float64
product of the same dequantized weights, at the edges of their 64-vector and
256- / 128- / 16-row tiles, and prompts (of several chunks, and of a
part of one) against the chunk-by-chunk path on the same weights (itself held to the oracle's
sequential forwards in test_gpu_prefill.py).

Tolerances: Q4_K and f16 weights enter the matrix cores exactly and the
vectors as 22-bit hi + lo pairs, so only f32 accumulation is left (a few
1e-7): 2e-6. Q6_K weights round sc * (q - 32) once to f16 (2^-12 at most,
1.4e-4 root mean square): 3e-4. A prompt's layers append f16 K/V rows, whose
half-ulp differences (2^-12) reach its last token: 1e-3, the paths' bar."""
import numpy as np
import pytest

import oracle as O
import synth
from g4hip import G4Error
from g4hip.decoder import BatchDecoder, E2BShape
from gpu_util import assert_close

pytestmark = pytest.mark.gpu

BAR = {"q4k": 2e-6, "q6k": 3e-4, "f16": 2e-6}


def _weights(wtype, seed, M, N):
    """Blocks as stored and their float64 values [M][N]."""
    if wtype == "f16":
        w = O.gen_normal_f16(seed, M * N, 0.0, 0.03)
        return w, O.np_f16_to_f32(w).astype(np.float64).reshape(M, N)
    b = (synth.q4k_centered if wtype == "q4k" else synth.q6k_wide)(seed, M * N // 256)
    deq = O.np_dequant_q4k if wtype == "q4k" else O.np_dequant_q6k
    return b, deq(b).astype(np.float64).reshape(M, N)


def _vectors(seed, T, N):
    X = O.gen_normal_f32(seed, T * N, 0.0, 1.5).reshape(T, N)
    X[T // 2] *= 40.0   # one vector of another scale, one with a huge element, one of zeros
    X[0, 3] = 3e4
    X[T - 1] = 0.0
    return X


def _ops(ctx, X):
    T, N = X.shape
    ops = ctx.alloc(ctx.prefill_operand_bytes(N, T))
    ctx.prefillPrep(ctx.from_numpy(X), 1, None, None, None, None, None, None, N, T, ops=ops)
    ctx.sync()
    return ops


@pytest.mark.parametrize("wtype,rows,N,T,split", [
    ("q4k", [2048, 256, 256], 1536, 65, 1),    # q/k/v, one vector past a tile
    ("q4k", [16], 1536, 1, 1),                 # the smallest
    ("q4k", [100, 33], 2048, 130, 1),          # rows that fill no tile, a padded segment
    ("q4k", [1536], 4096, 127, 16),            # o of a head-dim-512 layer, K split
    ("q6k", [1536], 2048, 64, 8),
    ("q6k", [257], 1536, 100, 2),              # one row past a 256-row group
    ("f16", [256], 1536, 129, 6),
    ("f16", [1536], 256, 70, 1),               # one super-block
    ("q4k", [4096, 512, 512], 1536, 700, 1),   # enough row groups and vectors for the wide row tiles
    ("q6k", [4096], 1536, 1030, 1),
])
def test_prefill_matmul(ctx, wtype, rows, N, T, split):
    WV = [_weights(wtype, 11 + i, M, N) for i, M in enumerate(rows)]
    X = _vectors(5, T, N)
    wops = ctx.alloc(ctx.prefill_weight_bytes(wtype, rows, N))
    Y = [ctx.zeros(split * T * M, np.float32) for M in rows]
    ks = ctx.prefillMatmul(wtype, [ctx.from_numpy(b) for b, _ in WV], Y, rows, N, _ops(ctx, X), T, wops, split)
    assert 1 <= ks <= split
    for (_, w), y, M in zip(WV, Y, rows):
        got = y.download(np.float32, ks * T * M).reshape(ks, T, M).astype(np.float64).sum(0)
        want = X.astype(np.float64) @ w.T
        assert np.all(np.isfinite(got))
        for v in sorted({0, T // 2, T - 1, min(63, T - 1), min(64, T - 1)}):
            assert O.rel_l2(got[v], want[v]) <= BAR[wtype], (M, v)
        assert O.rel_l2(got, want) <= BAR[wtype]


def _exact_blocks(wtype, seed, M, N):
    """Blocks whose operands f16 holds exactly (Q6_K: scales of at most 63), and their float64 values."""
    b = (synth.q4k_centered if wtype == "q4k" else synth.q6k_wide)(seed, M * N // 256)
    if wtype == "q6k":
        r = b.reshape(-1, 210)
        r[:, 192:208] = (r[:, 192:208].view(np.int8) // 2).view(np.uint8)
    return b, (O.np_dequant_q4k if wtype == "q4k" else O.np_dequant_q6k)(b).astype(np.float64).reshape(M, N)


def _step_ops(ctx, X):
    T, N = X.shape
    ops, xn = ctx.alloc(ctx.batch_operand_bytes(N, T)), ctx.zeros(T * N, np.float32)
    ctx.batchPrep(ctx.from_numpy(X), 1, None, None, None, None, xn, N, T, ops=ops)
    return ops, xn


@pytest.mark.parametrize("wtype", ["q4k", "q6k"])
def test_prefill_matmul_as_exact_as_the_step(ctx, wtype):
    """The same vectors through the ragged step's matmul and the prompt's: what is left with exact weights, f32
    accumulation, is of the same size (1.1: the two sum in different orders; measured 0.98 and 1.01)."""
    M, N, T = 2048, 1536, 64
    b, w = _exact_blocks(wtype, 51, M, N)
    X = O.gen_normal_f32(52, T * N).reshape(T, N)
    want = X.astype(np.float64) @ w.T
    db, y = ctx.from_numpy(b), ctx.zeros(T * M, np.float32)
    ops, xn = _step_ops(ctx, X)
    ctx.matmulSegmentsBatchPartial(wtype, xn, [db], [y], [M], N, T, 1, ops=ops)
    step = O.rel_l2(y.download(np.float32).reshape(T, M), want)
    ctx.prefillMatmul(wtype, [db], [y], [M], N, _ops(ctx, X), T, ctx.alloc(ctx.prefill_weight_bytes(wtype, [M], N)))
    got = O.rel_l2(y.download(np.float32).reshape(T, M), want)
    print(f"[prefill] {wtype}: step {step:.3e}, prompt {got:.3e}", flush=True)
    assert got <= 1.1 * step


@pytest.mark.parametrize("M,N,T,split", [
    (256, 1536, 129, 6),   # per-layer embeddings: the gate
    (1536, 256, 70, 1),    # and proj, one super-block
    (8960, 1536, 65, 1),   # the model projection, one vector past a tile
    (33, 2048, 1, 8),      # rows that fill no tile, one vector
])
@pytest.mark.parametrize("heavy", [False, True])
def test_prefill_f16_as_exact_as_the_matvec(ctx, M, N, T, split, heavy):
    """f16 rows with the vectors' third term against the f32 matvec of a step (1.1, the one vector 1.5: sums in
    different orders, over fewer of them), also where a few elements are far above the others."""
    wb, w = _weights("f16", 57, M, N)
    X = O.gen_normal_f32(58, T * N).reshape(T, N)
    if heavy:
        X *= np.exp(3.0 * np.random.default_rng(5).standard_normal(X.shape)).astype(np.float32)
    want = X.astype(np.float64) @ w.T
    dw, dx, y = ctx.from_numpy(wb), ctx.from_numpy(X), ctx.zeros(split * T * M, np.float32)
    ctx.matmulF16(dx, dw, y, M, N, T)
    step = O.rel_l2(y.download(np.float32, T * M).reshape(T, M), want)
    ops, lo = ctx.alloc(ctx.prefill_operand_bytes(N, T)), ctx.alloc(ctx.prefill_operand_lo_bytes(N, T))
    if N == 256:  # (gelu(20) is 20 in f32)
        one = ctx.from_numpy(np.full(T * N, 20.0, np.float32))
        ctx.prefillPleGated(one, 1, ctx.from_numpy(X / np.float32(20.0)), N, 0, None, T, ops=ops, ops_lo=lo)
        want = (np.float32(20.0) * (X / np.float32(20.0))).astype(np.float64) @ w.T
    else:
        ctx.prefillPrep(dx, 1, None, None, None, None, None, None, N, T, ops=ops, ops_lo=lo)
    ks = ctx.prefillMatmul("f16", [dw], [y], [M], N, ops, T, ctx.alloc(ctx.prefill_weight_bytes("f16", [M], N)),
                           split, ops_lo=lo)
    parts = y.download(np.float32, ks * T * M).reshape(ks, T, M)
    got = parts[0].copy()
    for p in parts[1:]:
        got += p
    got = O.rel_l2(got, want)
    print(f"[prefill] f16 {M}x{N} T={T} heavy={heavy}: matvec {step:.3e}, prompt {got:.3e}", flush=True)
    assert got <= (1.5 if T == 1 else 1.1) * step


@pytest.mark.parametrize("spread", [0, 20])  # of the gate rows' sizes from 32 to 32, in powers of two
def test_prefill_ffn_as_exact_as_the_step(ctx, spread):
    """The same through gate/up and down: the step scales the product per 32 rows, the prompt per 128."""
    M, N, T, H = 6144, 1536, 64, 1536
    gb, _ = _exact_blocks("q4k", 53, M, N)
    if spread:
        r = gb.reshape(M, -1, 144)
        d = r[:, :, 0:2].copy().view(np.float16)[..., 0].astype(np.float32)
        s = np.exp2(-spread * np.random.default_rng(4).random(M // 32)).repeat(32).astype(np.float32)
        d = (d * s[:, None]).astype(np.float16)
        r[:, :, 0:2] = d[..., None].view(np.uint8)
        r[:, :, 2:4] = (d.astype(np.float32) * 7.5).astype(np.float16)[..., None].view(np.uint8)
    g = O.np_dequant_q4k(gb).astype(np.float64).reshape(M, N)
    (ub, u), (db, d) = _exact_blocks("q4k", 54, M, N), _exact_blocks("q6k", 55, H, M)
    X = O.gen_normal_f32(56, T * N, 0.0, 0.5).reshape(T, N)
    a = X.astype(np.float64) @ g.T
    t = np.clip(0.7978845608028654 * a * (1 + 0.044715 * a * a), -15, 15)
    want = (0.5 * a * (1 + np.tanh(t)) * (X.astype(np.float64) @ u.T)) @ d.T
    dg, du, dd = (ctx.from_numpy(x) for x in (gb, ub, db))
    y = ctx.zeros(M // 256 * T * H, np.float32)

    def total(n):
        return O.rel_l2(y.download(np.float32, n * T * H).reshape(n, T, H).astype(np.float64).sum(0), want)

    ops, xn = _step_ops(ctx, X)
    prod = ctx.alloc(ctx.batch_sub_operand_bytes(M, T))
    ctx.gateUpGeluBatchOps(xn, ops, dg, du, None, prod, M, N, T)
    step = total(ctx.matmulSubBatchPartial(prod, dd, y, H, M, T, M // 768))
    prod = ctx.alloc(ctx.prefill_operand_bytes(M, T))
    wops = ctx.alloc(max(ctx.prefill_weight_bytes("q4k", [M, M], N), ctx.prefill_weight_bytes("q6k", [H], M)))
    ctx.prefillGateUp("q4k", dg, du, _ops(ctx, X), prod, M, N, T, wops)
    got = total(ctx.prefillMatmul("q6k", [dd], [y], [H], M, prod, T, wops, M // 768, product_ops=True))
    print(f"[prefill] ffn spread {spread}: step {step:.3e}, prompt {got:.3e}", flush=True)
    assert got <= 1.1 * step


@pytest.mark.parametrize("wtype", ["q4k", "q6k", "f16"])
@pytest.mark.parametrize("down", ["q4k", "q6k", "f16"])
def test_prefill_ffn(ctx, wtype, down):
    """gate/up -> GELU product -> down, over 90 vectors (a whole tile and a part of one)."""
    N, M, T = 1536, 512, 90
    (gb, g), (ub, u) = (_weights(wtype, s, M, N) for s in (21, 22))
    db, d = _weights(down, 23, 1536, M)
    X = O.gen_normal_f32(7, T * N, 0.0, 0.5).reshape(T, N)
    X[T // 2] *= 20.0
    X[T - 1] = 0.0
    wops = ctx.alloc(max(ctx.prefill_weight_bytes(wtype, [M, M], N), ctx.prefill_weight_bytes(down, [1536], M)))
    prod = ctx.alloc(ctx.prefill_operand_bytes(M, T))
    Y = ctx.zeros(2 * T * 1536, np.float32)
    ctx.prefillGateUp(wtype, ctx.from_numpy(gb), ctx.from_numpy(ub), _ops(ctx, X), prod, M, N, T, wops)
    ks = ctx.prefillMatmul(down, [ctx.from_numpy(db)], [Y], [1536], M, prod, T, wops, 2, product_ops=True)
    got = Y.download(np.float32, ks * T * 1536).reshape(ks, T, 1536).astype(np.float64).sum(0)
    x = X.astype(np.float64)
    a = x @ g.T
    t = np.clip(0.7978845608028654 * a * (1 + 0.044715 * a * a), -15, 15)
    want = (0.5 * a * (1 + np.tanh(t)) * (x @ u.T)) @ d.T
    # (the GELU's own f32 evaluation adds a few 1e-7 relative to the product's size; twice the weights' bar)
    bar = BAR[down] + 2 * BAR[wtype]
    assert np.all(np.isfinite(got))
    assert O.rel_l2(got, want) <= bar
    for v in (0, 63, 64):
        assert O.rel_l2(got[v], want[v]) <= bar, v


@pytest.mark.parametrize("T,parts", [(1, 1), (65, 3)])
def test_prefill_ple_gated(ctx, T, parts):
    """gelu(sum of the parts) * the layer's slice: the values, and their operand blocks through a product."""
    D, stride, off = 256, 768, 512
    gate = O.gen_normal_f32(31, parts * T * D, 0.0, 1.0).reshape(parts, T, D)
    ple = O.gen_normal_f32(32, T * stride).reshape(T, stride)
    out, ops = ctx.zeros(T * D, np.float32), ctx.alloc(ctx.prefill_operand_bytes(D, T))
    ctx.prefillPleGated(ctx.from_numpy(gate), parts, ctx.from_numpy(ple), stride, off, out, T, ops=ops)
    got = out.download(np.float32).reshape(T, D)
    a = gate.astype(np.float64).sum(0)
    t = np.clip(0.7978845608028654 * a * (1 + 0.044715 * a * a), -15, 15)
    want = 0.5 * a * (1 + np.tanh(t)) * ple[:, off:off + D]
    assert O.rel_l2(got, want) <= 2e-6
    wb, w = _weights("f16", 33, 48, D)
    y, wops = ctx.zeros(T * 48, np.float32), ctx.alloc(ctx.prefill_weight_bytes("f16", [48], D))
    ctx.prefillMatmul("f16", [ctx.from_numpy(wb)], [y], [48], D, ops, T, wops)
    assert O.rel_l2(y.download(np.float32).reshape(T, 48), got.astype(np.float64) @ w.T) <= BAR["f16"]


@pytest.mark.parametrize("layout,B,T,start", [
    ("uniform", 64, 65, 0),      # one row past a chunk
    ("uniform", 64, 300, 600),   # past the window
    ("real", 64, 131, 37),
    ("real", 7, 23, 0),          # odd chunks
    ("uniform", 1, 3, 5),        # (three chunks of few rows stay chunks)
    ("uniform", 1, 4, 5),
    ("uniform", 5, 16, 40),
    ("uniform", 64, 9, 0),       # one chunk: 16 and 32 of its rows, and all
    ("real", 64, 27, 700),
    ("uniform", 64, 33, 0),
    ("uniform", 20, 17, 500),
])
def test_wide_prefill_equals_chunks(ctx, layout, B, T, start):
    s = (E2BShape(n_layers=2, global_layers=(1,), vocab=4096) if layout == "uniform" else
         E2BShape.real(n_layers=4, n_unshared=2, global_layers=(1, 3), vocab=4096))
    d = BatchDecoder(ctx, [0] * B, s, seed=31, reserve=start + T + 2 * B, shared_pages=True, embed=True)
    assert d.wide_rows >= B
    toks = np.random.default_rng(3).integers(0, s.vocab, T).astype(np.uint32)

    def go(**kw):
        d.fill_kv(seed=32)
        row = d.prefill(toks, start, **kw)
        ctx.sync()
        kv = [p.download(np.uint16).view(np.float16).astype(np.float32) for L in d.layers
              for p in (L.k_cache, L.v_cache)]
        return (row, d.hidden.download(np.float32).reshape(B, -1), d.logits.download(np.float32).reshape(B, -1),
                d.tokens.download(np.uint32), d.seq_lens.download(np.uint32), kv)

    want = go(probe=lambda *a: None)  # chunk by chunk
    for rows in (d.wide_rows, max(B, 128 // B * B)):  # one pass, then several
        d.wide_rows = rows
        got = go()
        assert got[0] == want[0]
        n = got[0]
        assert_close(got[1][n], want[1][n], what="hidden")
        assert_close(got[2][n], want[2][n], what="logits")
        assert got[3][n] == O.argmax(got[2][n])
        assert np.array_equal(got[4], want[4])
        for a, b in zip(got[5], want[5]):
            assert_close(a, b, what="cache")


MIXES = {
    "q6k": lambda il, m: "q6k",
    "q4k": lambda il, m: "q4k",
    "mixed": lambda il, m: {"wq": "q4k", "wk": "q6k", "wv": "q4k", "wo": "q6k", "wdown": "q4k"}.get(m, "q6k"),
    "f16 q/k/v/o": lambda il, m: "f16" if m in ("wq", "wk", "wv", "wo") else "q4k" if m != "wdown" else "q6k",
    "f16 v, o of layer 1": lambda il, m: "f16" if m == "wv" or (m == "wo" and il) else "q4k",
}


@pytest.mark.parametrize("mix,shape,B,T", [
    ("q6k", {}, 64, 70), ("q4k", {}, 64, 129), ("mixed", {}, 16, 50), ("f16 q/k/v/o", {}, 64, 100),
    ("f16 v, o of layer 1", {"real": True}, 64, 90), ("mixed", {"hidden": 2048}, 64, 140),
    ("mixed", {"hidden": 2048, "real": True}, 32, 70),
    ("q4k", {"n_layers": 1, "global_layers": ()}, 64, 2100),  # past the rows of one pass
])
def test_wide_prefill_formats_and_widths(ctx, mix, shape, B, T):
    """A prompt in whole passes against its chunks, where the layers' formats differ, at the other hidden width, and
    past the rows of one pass: its last token's residual row and logits, and the K/V rows."""
    kw = dict(shape)
    make = E2BShape.real if kw.pop("real", False) else E2BShape
    s = make(**{"n_layers": 2, "global_layers": (1,), "vocab": 2048, **kw})
    d = BatchDecoder(ctx, [0] * B, s, seed=37, reserve=T + 2 * B, shared_pages=True, embed=True, wtypes=MIXES[mix])
    assert d.wide_rows >= B
    toks = np.random.default_rng(4).integers(0, s.vocab, T).astype(np.uint32)

    def go(**kw):
        d.fill_kv(seed=38)
        row = d.prefill(toks, 0, **kw)
        return [row, d.hidden.download(np.float32).reshape(B, -1)[row],
                d.logits.download(np.float32).reshape(B, -1)[row]] + [
                    p.download(np.uint16).view(np.float16).astype(np.float32) for L in d.layers
                    for p in (L.k_cache, L.v_cache)]

    want, got = go(probe=lambda *a: None), go()
    assert d.wide is not None and got[0] == want[0]
    for a, b in zip(got[1:], want[1:]):
        assert_close(a, b, what=f"{mix}, {T} tokens")


def _attn_case(ctx, hd, T, start, window, n_kv=1, short_ws=False):
    """Rows at start .. start + T - 1 of one scattered page list against the oracle's paged attention."""
    page, nq = 16, 8 * n_kv
    L = start + T
    pages = -(-L // page) + 2
    table = np.random.default_rng(L).permutation(pages).astype(np.int32)
    kp, vp = (O.gen_normal_f16(s, pages * page * n_kv * hd, 0.0, 1.0 if s == 42 else 0.25) for s in (41, 42))
    q = O.gen_normal_f32(43, T * nq * hd, 0.0, 0.5).reshape(T, nq * hd)
    lens = (start + 1 + np.arange(T)).astype(np.uint32)
    if T > 2:
        lens[-1] = lens[-2]   # a repeated row, as a padded chunk has
    p = ctx.paged_fused_params(T, nq, n_kv, hd, page, pages, pages * page, pages, window, 1e-6, 1e4, 0)
    out = ctx.zeros(T * nq * hd, np.float32)
    ws = None if short_ws else ctx.alloc(ctx.prefill_attn_workspace_bytes(p))
    ctx.prefillAttn(ctx.from_numpy(q), ctx.from_numpy(kp), ctx.from_numpy(vp), ctx.from_numpy(table),
                    ctx.from_numpy(lens), out, p, ws)
    got = out.download(np.float32).reshape(T, -1)
    for v in sorted({0, 1, 6, 7, 8, T // 2, T - 2, T - 1} & set(range(T))):
        want = O.attention_paged(q[v], kp, vp, table, page, nq, n_kv, hd, int(lens[v]), 1.0, window)
        # q and P enter as 22-bit pairs, exp2 is within 1e-5 relative: 4e-5
        assert_close(got[v], want, rel=4e-5, what=f"row {v}")


@pytest.mark.parametrize("hd", [256, 512])
@pytest.mark.parametrize("T,start,window", [
    (1, 0, 0), (7, 0, 0), (8, 0, 32), (9, 0, 0), (33, 0, 0), (65, 500, 512), (17, 31, 40), (40, 600, 512),
    (9, 3000, 0),      # few rows over a long cache: the window split over workgroups
    (300, 700, 0),
])
def test_prefill_attention(ctx, hd, T, start, window):
    _attn_case(ctx, hd, T, start, window)


def test_prefill_attention_two_kv_heads(ctx):
    _attn_case(ctx, 256, 21, 100, 64, n_kv=2)


def test_prefill_attention_without_workspace(ctx):
    _attn_case(ctx, 512, 9, 2000, 0, short_ws=True)


@pytest.mark.parametrize("hd", [256, 512])
@pytest.mark.parametrize("window", [0, 32])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_prefill_attention_non_finite_rows(ctx, hd, window, bad):
    """A non-finite V element reaches the rows whose window holds it, in its own dim, and no others: not those
    before it, nor (with a window) those past it, nor the rows of a tail step that repeats the last position."""
    page, nq, T, start = 16, 8, 45, 40
    L = start + T
    pages = -(-L // page)
    table = np.random.default_rng(3).permutation(pages).astype(np.int32)
    kp, vp = (O.gen_normal_f16(s, pages * page * hd, 0.0, 1.0 if s == 62 else 0.25) for s in (61, 62))
    q = O.gen_normal_f32(63, T * nq * hd, 0.0, 0.5).reshape(T, nq * hd)
    lens = (start + 1 + np.arange(T)).astype(np.uint32)
    poison = {start + 5: 3, start + 17: 130, 20: 7, L - 1: 200}  # position: dim
    rows = vp.view(np.float16).reshape(-1, hd)
    clean = rows.copy()
    for pos, d in poison.items():
        r = table[pos // page] * page + pos % page
        rows[r, d] = bad
        clean[r, d] = 0
    p = ctx.paged_fused_params(T, nq, 1, hd, page, pages, pages * page, pages, window, 1e-6, 1e4, 0)
    out = ctx.from_numpy(np.full(T * nq * hd, 7.0, np.float32))
    ctx.prefillAttn(ctx.from_numpy(q), ctx.from_numpy(kp), ctx.from_numpy(vp), ctx.from_numpy(table),
                    ctx.from_numpy(lens), out, p, ctx.alloc(ctx.prefill_attn_workspace_bytes(p)))
    got = out.download(np.float32).reshape(T, nq, hd)
    for v in range(T):
        n = int(lens[v])
        seen = {d for pos, d in poison.items() if (n - window if window else 0) <= pos < n}
        ok = [d for d in range(hd) if d not in seen]
        assert not np.isfinite(got[v][:, sorted(seen)]).any(), v
        want = O.attention_paged(q[v], kp, clean.view(np.uint16).reshape(-1), table, page, nq, 1, hd, n, 1.0, window)
        assert_close(got[v][:, ok], want.reshape(nq, hd)[:, ok], rel=4e-5, what=f"row {v}")


@pytest.mark.parametrize("sample", ["argmax", "topk"])
@pytest.mark.parametrize("B,T", [(64, 1), (64, 16), (64, 17), (64, 32), (64, 33), (20, 9), (20, 16), (20, 20)])
def test_one_chunk_spare_rows_repeat_the_last_token(ctx, B, T, sample):
    """The rows of a one-chunk prompt past its last token hold that token's residual row, logits and sample, also
    where the step ran over 16 or 32 rows only; nothing of an earlier step is left in them."""
    s = E2BShape(n_layers=1, global_layers=(), vocab=1024)
    d = BatchDecoder(ctx, [0] * B, s, seed=33, reserve=2 * B + 40, shared_pages=True, embed=True)
    for buf in (d.hidden, d.logits, d.topk):
        buf.upload(np.full(buf.nbytes // 4, np.nan, np.float32))
    d.tokens.upload(np.full(B, 4000000000, np.uint32))
    toks = np.random.default_rng(T).integers(0, s.vocab, T).astype(np.uint32)
    n = d.prefill(toks, 7, sample=sample)
    assert n == T - 1
    outs = [d.hidden.download(np.uint32).reshape(B, -1), d.logits.download(np.uint32).reshape(B, -1)]
    if sample == "topk":
        outs.append(d.topk.download(np.uint32).reshape(B, -1))
        assert np.array_equal(d.tokens.download(np.uint32), np.concatenate([toks, np.repeat(toks[-1], B - T)]))
    else:
        outs.append(d.tokens.download(np.uint32).reshape(B, 1))
    assert np.all(np.isfinite(outs[1].view(np.float32)))
    for out in outs:
        assert np.array_equal(out[n:], np.repeat(out[n:n + 1], B - n, axis=0))
    assert np.array_equal(d.seq_lens.download(np.uint32), 8 + np.minimum(np.arange(B), T - 1))


@pytest.mark.parametrize("words,src,first,count", [(1, 3, 4, 60), (255, 0, 1, 1), (257, 9, 0, 9), (1536, 15, 16, 48)])
def test_repeat_row(ctx, words, src, first, count):
    rows = max(src + 1, first + count) + 1
    x = np.random.default_rng(words).integers(0, 2 ** 32, (rows, words), dtype=np.uint32)
    d = ctx.from_numpy(x)
    ctx.repeatRow(d, words, src, first, count)
    x[first:first + count] = x[src]
    assert np.array_equal(d.download(np.uint32).reshape(rows, words), x)
    with pytest.raises(G4Error, match="repeatRow"):
        ctx.repeatRow(d, words, first, first, count)


def test_wide_buffers_come_with_the_first_long_prompt(ctx):
    """A decoder whose prompts fit a chunk holds no buffers of a whole-prompt pass; a longer prompt brings them, a
    longer one again replaces them, and what came before changes no result."""
    B, s = 32, E2BShape.real(n_layers=3, n_unshared=2, global_layers=(1,), vocab=2048)

    def decoder():
        return BatchDecoder(ctx, [0] * B, s, seed=35, reserve=700, shared_pages=True, embed=True)

    def prompt(d, T):
        row = d.prefill(np.random.default_rng(T).integers(0, s.vocab, T).astype(np.uint32), 0)
        return d.hidden.download(np.uint32), d.logits.download(np.uint32), d.tokens.download(np.uint32), row

    d = decoder()
    assert d.wide_rows == 704 and d.wide is None
    prompt(d, 20)
    prompt(d, 64)  # (two chunks of 32)
    assert d.wide is None and d.wide_cap == 0
    caps = []
    for T in (70, 100, 333, 699, 70):
        got = prompt(d, T)
        caps.append(d.wide_cap)
        for a, b in zip(got, prompt(decoder(), T)):
            assert np.array_equal(a, b), T
    assert caps == [96, 192, 384, 704, 704]
