"""GPU parity of the paged batch attention at head dim 512 (Gemma-4-E2B's global
layers in the ragged step) against the oracle's paged attention: its
matrix-core form at the edges of its 64-position steps and of chunks of one,
two, three and more of them, with windows, two KV heads and empty sequences,
and the VALU form below its ranges (windows under 1024 positions, fewer than
64 positions per CU in all) and past them (65 sequences). The exponentials are
the hardware exp2 (1e-5 relative at most): 4e-5. The sequences share the pool's
pages, each in an order of its own."""
import numpy as np
import pytest

import oracle as O
from gpu_util import assert_close

pytestmark = pytest.mark.gpu

HD, PAGE = 512, 16


def _run(ctx, lens, cap, window, n_kv, ops=None):
    """(out [B][8 n_kv * 512], the oracle's row of a sequence)."""
    nq, B = 8 * n_kv, len(lens)
    per = -(-cap // PAGE)
    pages = per + 3
    rng = np.random.default_rng(B)
    table = np.stack([rng.permutation(pages)[:per] for _ in range(B)]).astype(np.int32)
    kp, vp = (O.gen_normal_f16(s, pages * PAGE * n_kv * HD, 0.0, 1.0 if s == 52 else 0.2) for s in (51, 52))
    q = O.gen_normal_f32(53, B * nq * HD, 0.0, 0.5).reshape(B, nq * HD)
    p = ctx.paged_params(B, nq, n_kv, HD, PAGE, per, cap, pages, 1.0, window)
    out = ctx.from_numpy(np.full(B * nq * HD, np.nan, np.float32))  # (a row left out is not finite)
    ctx.pagedAttnDecode(ctx.from_numpy(q), ctx.from_numpy(kp), ctx.from_numpy(vp), ctx.from_numpy(table),
                        ctx.from_numpy(np.array(lens, np.uint32)), out, p, ctx.alloc(ctx.paged_workspace_bytes(p)),
                        ops=ops)
    return (out.download(np.float32).reshape(B, -1),
            lambda b: O.attention_paged(q[b], kp, vp, table[b], PAGE, nq, n_kv, HD, lens[b], 1.0, window))


EDGES = [1, 63, 64, 65, 0, 127, 128, 129, 191, 192, 193, 255, 256, 257]


@pytest.mark.parametrize("lens,cap,window,n_kv", [
    ([1], 4, 0, 1),                                # the VALU form
    ([63, 64, 65, 1, 0, 129, 600], 603, 0, 1),
    ([700, 3, 512, 513], 703, 640, 1),
    ([40, 41, 2000], 2003, 40, 2),
    ([9] * 65, 12, 0, 1),
    (EDGES + [1022, 1023], 1023, 0, 1),            # a window one short of the matrix cores'
    (EDGES + [1023], 1024, 0, 1),                  # one sequence short of them
    (EDGES + [1023, 1024], 1024, 0, 1),            # chunks of one step
    (EDGES[:7] + [2099], 2100, 0, 1),              # two
    (EDGES + [383, 384, 385, 1], 2690, 0, 1),      # three, one round
    (list(range(1, 1300, 25)), 1279, 0, 1),        # three, two rounds
    (EDGES * 2 + [4000, 0, 511, 512, 513], 4001, 0, 1),  # by four rounds
    (EDGES[:9] + [1023, 1024, 1025, 1087, 1088, 2500, 2999], 3000, 1024, 1),
    ([40, 41, 2000, 0, 64], 2003, 0, 2),
])
def test_paged_attention_head_dim_512(ctx, lens, cap, window, n_kv):
    B = len(lens)
    got, want = _run(ctx, lens, cap, window, n_kv)
    for b in range(B) if B <= 40 else sorted(set(range(0, B, 7)) | {1, 2, B - 1}):
        if lens[b] == 0:
            assert not got[b].any(), b
        else:
            assert_close(got[b], want(b), rel=4e-5, what=f"sequence {b} of length {lens[b]}")
    assert np.all(np.isfinite(got))


@pytest.mark.parametrize("lens,cap", [(EDGES[:7] + [700], 710), (EDGES + [1023, 1024, 600], 1024)])
def test_operand_blocks(ctx, lens, cap):
    """The merge's operand blocks of the o projection hold the output it stores: f16 hi + lo of x * 2^e, 2^e from the
    256 elements' largest (to 2^13 .. 2^14): within 2^-22 of that largest, in both forms."""
    B, nsb, ntv = len(lens), 8 * HD // 256, 1 if len(lens) <= 16 else 2
    ops = ctx.zeros(ctx.batch_operand_bytes(8 * HD, B), np.uint8)
    got, _ = _run(ctx, lens, cap, 0, 1, ops)
    blk = ops.download(np.uint8).reshape(nsb, ntv * (16384 + 1024 + 64))
    main = blk[:, :ntv * 16384].copy().view(np.float16).reshape(nsb, ntv, 8, 2, 4, 16, 8).astype(np.float64)
    inv = blk[:, ntv * 17408:].copy().view(np.float32).reshape(nsb, ntv, 1, 1, 16, 1).astype(np.float64)
    val = ((main[:, :, :, 0] + main[:, :, :, 1]) * inv).transpose(1, 4, 0, 2, 3, 5).reshape(16 * ntv, 8 * HD)[:B]
    am = np.abs(got.astype(np.float64)).reshape(B, nsb, 256).max(-1, keepdims=True)
    assert np.all(np.abs(val - got).reshape(B, nsb, 256) <= am * 2.0 ** -22)
    assert np.all(np.isfinite(got)) and got.any()
