"""GPU parity of the paged batch attention at head dim 512 on the matrix cores
(Gemma-4-E2B's global layers in the ragged step) against the oracle's paged
attention, at the edges of its 64-position steps and of its chunks, with
windows, two KV heads, empty sequences, and past its ranges (65 sequences,
short windows: the VALU kernel). q and P enter as f16 hi + lo pairs (22 bits) and the
exponentials are the hardware exp2 (1e-5 relative at most): 4e-5; the operand
blocks of the o projection hold the same 22 bits."""
import numpy as np
import pytest

import oracle as O
from gpu_util import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,window,n_kv", [
    ([1], 0, 1),                         # (windows of at most 512 positions: the VALU kernel)
    ([63, 64, 65, 1, 0, 129, 600], 0, 1),
    ([700, 3, 512, 513], 640, 1),
    ([40, 41, 2000], 0, 2),
    ([40, 41, 2000], 40, 2),
    (list(range(1, 1300, 25)), 0, 1),    # chunks of several steps, more of them than CUs
    ([9] * 65, 0, 1),
])
def test_paged_attention_head_dim_512(ctx, lens, window, n_kv):
    hd, page, nq, B = 512, 16, 8 * n_kv, len(lens)
    max_len = max(lens) + 3
    per = -(-max_len // page)
    pages = B * per
    table = np.random.default_rng(B).permutation(pages).astype(np.int32).reshape(B, per)
    kp, vp = (O.gen_normal_f16(s, pages * page * n_kv * hd, 0.0, 1.0 if s == 52 else 0.2) for s in (51, 52))
    q = O.gen_normal_f32(53, B * nq * hd, 0.0, 0.5).reshape(B, nq * hd)
    p = ctx.paged_params(B, nq, n_kv, hd, page, per, max_len, pages, 1.0, window)
    ws = ctx.alloc(ctx.paged_workspace_bytes(p))
    out = ctx.zeros(B * nq * hd, np.float32)
    ctx.pagedAttnDecode(ctx.from_numpy(q), ctx.from_numpy(kp), ctx.from_numpy(vp), ctx.from_numpy(table),
                        ctx.from_numpy(np.array(lens, np.uint32)), out, p, ws)
    got = out.download(np.float32).reshape(B, -1)
    for b in sorted(set(range(0, B, 7)) | {1, B - 1} & set(range(B))):
        if lens[b] == 0:
            assert not got[b].any()
            continue
        want = O.attention_paged(q[b], kp, vp, table[b], page, nq, n_kv, hd, lens[b], 1.0, window)
        assert_close(got[b], want, rel=4e-5, what=f"sequence {b} of length {lens[b]}")
