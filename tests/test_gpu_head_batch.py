"""GPU parity of the tall Q6_K matmul (the LM head over up to 32 vectors): rows
at both ends and a sample of the others against a float64 product of the same
dequantized weights, every output finite and the same from call to call, with whole and short last tiles of 16 rows, both widths,
vector counts on both sides of a 16-vector tile, and the softcap. The weight
operand rounds sc * (q - 32) once to f16 (2^-12 at most, 1.4e-4 root mean
square): 3e-4, of the products. Behind the softcap that holds while its slope
is near 1, so the vector of another scale is left out there: products of ten
times the cap would leave, on the few outputs that do not saturate, an error
of 1.4e-4 of those products (3.5e-4 of the outputs' norm)."""
import numpy as np
import pytest

import oracle as O
import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,B,cap", [
    (65536, 1536, 16, 30.0),
    (65536 + 5, 1536, 2, 0.0),     # a last tile of 5 rows; rows not a multiple of 4
    (65536 + 16, 1536, 17, 30.0),
    (65536 + 7, 2048, 32, 0.0),
    (65536 + 12, 2048, 9, 30.0),
])
def test_tall_q6k_matmul(ctx, M, N, B, cap):
    b = synth.q6k_wide(71, M * N // 256)
    X = O.gen_normal_f32(72, B * N, 0.0, 0.3).reshape(B, N)
    if not cap:
        X[B // 2] *= 30.0
    ops, xn, y = ctx.alloc(ctx.batch_operand_bytes(N, B)), ctx.zeros(B * N, np.float32), ctx.zeros(B * M, np.float32)
    ctx.batchPrep(ctx.from_numpy(X), 1, None, None, None, None, xn, N, B, ops=ops)
    at = 4 if M % 4 else 0  # (weights are 4-byte aligned)
    buf = ctx.alloc(b.nbytes + at).upload(b, at)
    w = buf.offset(at)

    def call():
        y.upload(np.full(B * M, np.nan, np.float32))
        assert ctx.matmulSegmentsBatchPartial("q6k", xn, [w], [y], [M], N, B, 1, ops=ops, softcap=cap) == 1
        return y.download(np.float32).reshape(B, M)

    got = call()
    assert np.all(np.isfinite(got))
    for _ in range(2):  # the sums' order is fixed: every output again, bit for bit
        assert np.array_equal(call().view(np.uint32), got.view(np.uint32))
    rows = np.unique(np.concatenate([np.arange(40), np.arange(M - 40, M),
                                     np.random.default_rng(1).integers(0, M, 200)]))
    w = O.np_dequant_q6k(b.reshape(M, -1)[rows].reshape(-1)).astype(np.float64).reshape(len(rows), N)
    want = X.astype(np.float64) @ w.T
    if cap:
        want = np.tanh(np.clip(want / cap, -15, 15)) * cap
    for v in range(B):
        assert O.rel_l2(got[v, rows], want[v]) <= 3e-4, v
