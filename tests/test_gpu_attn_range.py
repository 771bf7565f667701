"""The matrix-core attentions of the paged batch (head dim 512) and of a prompt
(256 and 512) over the range of f32 queries and probabilities, against float64:
a dominant key whose V is small (the other probabilities, down to e^-20, carry
the result), query elements past f16's largest, tiny queries, and a key whose
score is -infinity through an infinite element (left out, as exp(-inf) is 0).

Bound: q and P enter as 22-bit pairs (2^-23 relative each), the scores (up to
16 here) and their exponents are f32 (2^-20 absolute, 2^-21 rounded): 2e-6."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BAR, PAGE, NQ, L = 2e-6, 16, 8, 1100


def _inputs(kind, hd, T):
    """q [T][8][hd], K and V [L][hd] (f16), as positions."""
    rng = np.random.default_rng(len(kind) + hd)
    q = rng.standard_normal((T, NQ, hd)).astype(np.float32)
    k = (rng.standard_normal((L, hd)) / np.sqrt(hd)).astype(np.float16)
    v = rng.standard_normal((L, hd)).astype(np.float16)
    if kind == "sink":
        q[:] = q[0, 0] + 0.01 * q
        k[1] = (14.0 * q[0, 0] / (q[0, 0] @ q[0, 0])).astype(np.float16)
        k *= np.float16(0.25)
        k[1] *= np.float16(4.0)
        v[1] *= np.float16(0.01)
    elif kind == "large":
        q[..., 3] = 1e5
        q[..., hd - 2] = -3e5
        k[:, 3] = (rng.standard_normal(L) * 2e-5).astype(np.float16)
        k[:, hd - 2] = (rng.standard_normal(L) * 5e-6).astype(np.float16)
    elif kind == "tiny":
        q *= np.float32(1e-6)
        k = (k.astype(np.float32) * 1e4).astype(np.float16)
        q *= np.float32(100.0)
    else:
        q[..., 5] = -np.abs(q[..., 5]) - 0.1
        k[700, 5] = np.inf
    return q, k, v


def _want(q, k, v, n):
    with np.errstate(invalid="ignore"):
        s = q.astype(np.float64) @ k[:n].astype(np.float64).T
    p = np.exp(s - s.max(-1, keepdims=True))
    return p @ v[:n].astype(np.float64) / p.sum(-1, keepdims=True)


def _pool(x, table, hd):
    """Positions to pool rows."""
    pool = np.zeros((table.size * PAGE, hd), np.float16)
    for i, pg in enumerate(table):
        rows = x[i * PAGE:(i + 1) * PAGE]
        pool[pg * PAGE:pg * PAGE + len(rows)] = rows
    return pool


def _check(got, want, what):
    assert np.all(np.isfinite(got)), what
    r = O.rel_l2(got.reshape(-1), want.reshape(-1))
    assert r <= BAR, (what, r)


KINDS = ["sink", "large", "tiny", "left out"]


@pytest.mark.parametrize("kind", KINDS)
def test_paged_512(ctx, kind):
    hd, B = 512, 16  # (fewer positions in all take the VALU form)
    lens = [L, 800, 705, 900] * 4
    q, k, v = _inputs(kind, hd, B)
    per = -(-L // PAGE)
    order = np.random.default_rng(2).permutation(B * per).astype(np.int32).reshape(B, per)
    kp, vp = np.zeros((B * per * PAGE, hd), np.float16), np.zeros((B * per * PAGE, hd), np.float16)
    for b in range(B):
        for i, pg in enumerate(order[b]):
            n = len(k[i * PAGE:(i + 1) * PAGE])
            kp[pg * PAGE:pg * PAGE + n], vp[pg * PAGE:pg * PAGE + n] = k[i * PAGE:][:n], v[i * PAGE:][:n]
    p = ctx.paged_params(B, NQ, 1, hd, PAGE, per, L, B * per, 1.0, 0)
    out = ctx.from_numpy(np.full(q.size, 7.0, np.float32))
    ctx.pagedAttnDecode(ctx.from_numpy(q), ctx.from_numpy(kp.view(np.uint16)), ctx.from_numpy(vp.view(np.uint16)),
                        ctx.from_numpy(order), ctx.from_numpy(np.array(lens, np.uint32)), out, p,
                        ctx.alloc(ctx.paged_workspace_bytes(p)))
    got = out.download(np.float32).reshape(q.shape)
    for b in range(B):
        _check(got[b], _want(q[b], k, v, lens[b]), (kind, b))


@pytest.mark.parametrize("hd", [256, 512])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("T", [11, 300])  # windows split over workgroups, and whole
def test_prompt(ctx, kind, hd, T):
    q, k, v = _inputs(kind, hd, T)
    table = np.random.default_rng(3).permutation(-(-L // PAGE)).astype(np.int32)
    lens = (L - T + 1 + np.arange(T)).astype(np.uint32)
    p = ctx.paged_fused_params(T, NQ, 1, hd, PAGE, table.size, L, table.size, 0, 1e-6, 1e4, 0)
    out = ctx.from_numpy(np.full(q.size, 7.0, np.float32))
    ctx.prefillAttn(ctx.from_numpy(q), ctx.from_numpy(_pool(k, table, hd).view(np.uint16)),
                    ctx.from_numpy(_pool(v, table, hd).view(np.uint16)), ctx.from_numpy(table), ctx.from_numpy(lens),
                    out, p, ctx.alloc(ctx.prefill_attn_workspace_bytes(p)))
    got = out.download(np.float32).reshape(q.shape)
    for t in sorted({0, 1, 7, 8, T // 2, T - 1}):
        _check(got[t], _want(q[t], k, v, int(lens[t])), (kind, t))
