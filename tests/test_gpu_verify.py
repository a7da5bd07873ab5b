"""GPU: several activation vectors over one weight matrix (verify), M = 2..16.

The vectors sit in the rows of the matrix-core operand, four to a group, and a
launch is cut into K slices of four blocks: sizes here are the edges of the
groups (M = 2, 4, 5, 8, 9, 12, 13, 16), of the 16-row tiles, and of the slices
and their two-block stages (1 to 9 blocks, whole and short last slices).  Odd
Q6_K block counts run their even and odd rows as two matrices of twice the row
stride, either row count parity.

Bar: every row within 2e-5 * sum|w*x| of the f64 dot; non-finite rows in the
category that per-weight f32 products give.
"""
import numpy as np
import pytest

import crafted
import oracle_lib as O
import quantize
import si_hip
from test_gpu_parity import _category, assert_dot_close, log, same_bits

pytestmark = pytest.mark.gpu

SIZES = [(1, 256, 2), (15, 512, 3), (17, 768, 4), (33, 1024, 5), (16, 1280, 8), (47, 1536, 9),
         (3, 1792, 12), (130, 2048, 13), (256, 2304, 16), (1001, 5376, 6), (4100, 2560, 16),
         (2, 11008, 16), (999, 17152, 7)]


@pytest.mark.parametrize("t", [12, 13, 14])
@pytest.mark.parametrize("rows,cols,batch", SIZES)
def test_verify_edges(hip_ctx, t, rows, cols, batch):
    log(f"verify t={t} {rows}x{cols} M={batch}")
    w = si_hip.synth_matrix(t, seed=rows + cols + t, rows=rows, cols=cols, threads=8)
    X = si_hip.synth_normal(rows * 3 + cols + batch, batch * cols).reshape(batch, cols).copy()
    X[:, ::97] *= np.float32(300.0)  # a few large channels
    X[batch - 1, :256] = 0.0
    W = hip_ctx.upload_quant_weight_private(w, t)
    try:
        outs = [o.copy() for o in hip_ctx.gguf_quant_matmul_many_weight(W, rows, cols, batch, X)]
        for b in range(batch):
            _, y64, ab = O.matvec(t, w, rows, cols, X[b], threads=8)
            assert_dot_close(outs[b], y64, ab, what=f"vector {b}")
        again = hip_ctx.gguf_quant_matmul_many_weight(W, rows, cols, batch, X)
        assert all(same_bits(a, o) for a, o in zip(again, outs))
    finally:
        W.free()


@pytest.mark.parametrize("t", [12, 13, 14])
@pytest.mark.parametrize("rows,cols", [(1, 256), (16, 512), (17, 768), (300, 1024), (4097, 1280),
                                       (260, 3584), (8192, 4096), (33, 4352), (2100, 4608),
                                       (1700, 5120), (1400, 6144), (28000, 512), (4112, 2560)])
def test_two_vectors_in_whole_rows(hip_ctx, t, rows, cols):
    """Two vectors of short rows, one launch of whole rows: odd and even block
    counts, one tile to several a workgroup, both sides of the lines to the
    vectors-in-rows kernel; rounded blocks and blocks on the exact path in either
    vector."""
    log(f"two vectors t={t} {rows}x{cols}")
    w = si_hip.synth_matrix(t, seed=rows + cols + 3 * t, rows=rows, cols=cols, threads=8)
    X = si_hip.synth_normal(rows + 2 * cols, 2 * cols).reshape(2, cols).copy()
    X[:, ::97] *= np.float32(300.0)
    X[0, :256] = 0.0
    X[1, cols - 200:] *= np.float32(1e-7)
    X[1, cols - 256] = 1.0
    W = hip_ctx.upload_quant_weight_private(w, t)
    try:
        outs = [o.copy() for o in hip_ctx.gguf_quant_matmul_many_weight(W, rows, cols, 2, X)]
        for b in range(2):
            _, y64, ab = O.matvec(t, w, rows, cols, X[b], threads=8)
            assert_dot_close(outs[b], y64, ab, what=f"vector {b}")
        again = hip_ctx.gguf_quant_matmul_many_weight(W, rows, cols, 2, X)
        assert all(same_bits(a, o) for a, o in zip(again, outs))
        X[0, cols - 1], X[1, 3] = np.inf, np.nan  # each in one vector's block alone
        X[1, cols - 1] = np.float32(1e35)
        outs = hip_ctx.gguf_quant_matmul_many_weight(W, rows, cols, 2, X)
        for b in range(2):
            y32, _, _ = O.matvec(t, w, rows, cols, X[b], threads=8)
            assert np.array_equal(_category(outs[b]), _category(y32)), f"vector {b}"
    finally:
        W.free()


@pytest.mark.parametrize("t,rows,cols", [(12, 37, 1792), (13, 37, 1792), (14, 37, 1792),
                                         (14, 38, 2304), (14, 38, 2560)])
def test_verify_special_blocks(hip_ctx, t, rows, cols):
    """Huge, subnormal and side blocks within the bound, and one infinite or NaN
    activation in the first and the last block of a vector (its neighbours'
    rows stay finite)."""
    batch = 6
    w = si_hip.synth_matrix(t, seed=77 * t + cols, rows=rows, cols=cols, threads=8)
    X = si_hip.synth_normal(78 * t + rows, batch * cols).reshape(batch, cols).copy()
    X[1, 100:140] = np.float32(3e30)
    X[2, 300] = np.float32(1e-9)
    X[2, 512:768] = np.float32(1e-41)
    X[3, cols - 1] = np.inf
    X[4, 0] = np.nan
    X[5, 3] = -np.inf
    W = hip_ctx.upload_quant_weight_private(w, t)
    try:
        outs = hip_ctx.gguf_quant_matmul_many_weight(W, rows, cols, batch, X)
        for b in range(batch):
            y32, y64, ab = O.matvec(t, w, rows, cols, X[b], threads=8)
            assert np.array_equal(_category(outs[b]), _category(y32)), f"vector {b}"
            if b < 3:
                assert_dot_close(outs[b], y64, ab, what=f"vector {b}")
    finally:
        W.free()


@pytest.mark.parametrize("t", [12, 13])
@pytest.mark.parametrize("rows,cols,batch", [(480, 512, 1), (400, 5120, 1), (17408, 5120, 1),
                                             (330, 2816, 2), (400, 8192, 2), (400, 5120, 4),
                                             (330, 2816, 5), (400, 5120, 16)])
def test_cancelling_terms(hip_ctx, t, rows, cols, batch):
    """A nearly constant vector against weights quantised from zero-mean ones, so
    that a block's scale and minimum terms are some seventy times its dot: the error
    stays what the f32 rounding of the partial sums makes it, at most 2^-25 of a sum
    and of either sign, under 2^-24 of the blocks' |dots| over the rows.  (With the
    terms in f32 it is their size that counts.)"""
    log(f"cancelling terms t={t} {rows}x{cols} M={batch}")
    rng = np.random.default_rng(rows + 9 * cols + t)
    base = min(rows, 480)
    w = quantize.quantize(t, 0.02 * rng.standard_normal((base, cols)))
    scales, mins = quantize.terms(t, w)
    assert np.median(np.abs(scales - mins) / (scales + mins)) < 0.02
    X = (1.0 + 1e-3 * rng.standard_normal((batch, cols))).astype(np.float32)
    dq = O.dequantize(t, w, base * cols).reshape(base, cols // 256, 256).astype(np.float64)
    X64 = X.astype(np.float64).reshape(batch, cols // 256, 256)
    reps = -(-rows // base)
    W = hip_ctx.upload_quant_weight_private(
        np.tile(w.reshape(base, -1), (reps, 1))[:rows].reshape(-1), t)
    try:
        if batch == 1:
            outs = [hip_ctx.gguf_quant_matvec_weight(W, rows, cols, X[0])]
        else:
            outs = hip_ctx.gguf_quant_matmul_many_weight(W, rows, cols, batch, X)
        for b in range(batch):
            dots = (dq * X64[b]).sum(2)
            err = outs[b][:base].astype(np.float64) - dots.sum(1)
            rms = np.sqrt(np.mean(err ** 2)) / np.sqrt(np.mean(np.abs(dots).sum(1) ** 2))
            assert rms <= 2.0 ** -24, f"vector {b}: {rms:.2e}"
    finally:
        W.free()


@pytest.mark.parametrize("rows,cols,start", [(3, 256, 1), (64, 1280, 3), (129, 6912, 5),
                                             (4097, 1280, 1), (40, 1280, 2)])
def test_q6k_rows_off_a_word(hip_ctx, rows, cols, start):
    """Q6_K matrices that start inside another one: with an odd block count an odd
    row starts 2 bytes off a word, where the copies into LDS cannot."""
    log(f"q6k rows {start}..{start + rows} of {cols}")
    total, rb = rows + start + 1, cols // 256 * 210
    w = si_hip.synth_matrix(14, seed=rows + cols, rows=total, cols=cols, threads=8)
    part = w[start * rb:(start + rows) * rb]
    X = si_hip.synth_normal(rows + 7 * cols, 5 * cols).reshape(5, cols).copy()
    ref = [O.matvec(14, part, rows, cols, X[b], threads=8)[1:] for b in range(5)]
    W = hip_ctx.upload_quant_weight_private(w, 14)
    V = W.view(start * rb, rows * rb, 14)
    try:
        y = hip_ctx.gguf_quant_matvec_tensor_rows(W, (cols, total), start, rows, X[0])
        assert_dot_close(y, *ref[0], what="row range")
        _, logits = hip_ctx.gguf_quant_matvec_argmax_weight(V, rows, cols, X[0])
        assert_dot_close(logits, *ref[0], what="head")
        for batch in (2, 5):
            outs = hip_ctx.gguf_quant_matmul_many_weight(V, rows, cols, batch, X[:batch])
            for b in range(batch):
                assert_dot_close(outs[b], *ref[b], what=f"vector {b} of {batch}")
        both = hip_ctx.gguf_quant_matvec_many_weights([V, V], [rows, rows], cols, X[0])
        for y in both:
            assert_dot_close(y, *ref[0], what="group")
    finally:
        V.free()
        W.free()


@pytest.mark.parametrize("t,cols", [(12, 2048), (13, 2304), (14, 2048), (14, 2304)])
@pytest.mark.parametrize("batch", [2, 4, 5, 16])
def test_verify_dot_on_small_activations(hip_ctx, t, cols, batch):
    """A dot that eight side elements a block carry keeps f32 precision: they may
    cost 2^-21 of sum|w*x|, and each slice of four blocks and the sum over the
    slices round once to f32 (2^-24).  Two vectors of short rows run in the
    one-vector kernel's form, which holds them to 4e-6."""
    rows = 20
    w, x = crafted.small_dot(t, rows, cols)
    _, y64, ab = O.matvec(t, w, rows, cols, x, threads=8)
    assert ab.min() > 0.0
    slices = (cols // 256 + 4) // 4
    W = hip_ctx.upload_quant_weight_private(w, t)
    try:
        outs = hip_ctx.gguf_quant_matmul_many_weight(W, rows, cols, batch, np.stack([x] * batch))
        for b in range(batch):
            tol = 4e-6 if batch == 2 and cols // 256 % 2 == 0 or batch == 2 and t != 14 else 2.0 ** -21
            assert_dot_close(outs[b], y64, ab, tol + (slices + 1) * 2.0 ** -24, f"vector {b}")
    finally:
        W.free()


@pytest.mark.parametrize("t,nb", [(t, nb) for t in (12, 13) for nb in (1, 4, 5, 6, 9, 13, 17)] +
                         [(14, 5), (14, 6), (14, 9)])
@pytest.mark.parametrize("batch", [3, 7])
def test_verify_redone_slices(hip_ctx, t, nb, batch):
    """Vectors whose every slice is redone in the reduce, beside an ordinary one, at
    block counts that leave the last slice one to four blocks."""
    rows, cols = 301, 256 * nb
    log(f"verify redone slices t={t} nb={nb} M={batch}")
    w = crafted.zero_weight_matrix(t, rows, cols, seed=nb + t)
    X = np.stack([crafted.crafted_x(cols, "tiny", seed=nb + b) for b in range(batch)])
    X[1] = si_hip.synth_normal(nb, cols)
    W = hip_ctx.upload_quant_weight_private(w, t)
    try:
        outs = hip_ctx.gguf_quant_matmul_many_weight(W, rows, cols, batch, X)
        for b in range(batch):
            _, y64, ab = O.matvec(t, w, rows, cols, X[b], threads=8)
            assert_dot_close(outs[b], y64, ab, 1e-6, f"vector {b}")
    finally:
        W.free()


@pytest.mark.parametrize("t,rows,nb", [(12, 65573, 128), (13, 65573, 128), (14, 65573, 128),
                                       (14, 65573, 127), (14, 65574, 127)])
def test_verify_in_several_row_ranges(hip_ctx, t, rows, nb):
    """Sixteen vectors whose partial sums fill the scratch three times over: the
    ranges are 32768 rows and a ragged rest (an odd and an even one where the rows
    run in pairs).  The matrix is 64 rows over and over, so every row is, bit for
    bit, that of a matrix of those alone, one range."""
    cols, period, batch = 256 * nb, 64, 16
    log(f"verify in ranges t={t} {rows}x{cols}")
    small = si_hip.synth_matrix(t, seed=nb + t, rows=period, cols=cols, threads=8)
    row_bytes = small.size // period
    big = np.tile(small, -(-rows // period))[:rows * row_bytes]
    X = si_hip.synth_normal(nb, batch * cols).reshape(batch, cols).copy()
    X[3, 300:600] *= np.float32(1e-6)
    X[5, cols - 1] = np.inf
    S, W = (hip_ctx.upload_quant_weight_private(m, t) for m in (small, big))
    del big
    try:
        want = [o.copy() for o in hip_ctx.gguf_quant_matmul_many_weight(S, period, cols, batch, X)]
        outs = hip_ctx.gguf_quant_matmul_many_weight(W, rows, cols, batch, X)
        for b in range(batch):
            assert same_bits(outs[b], np.tile(want[b], -(-rows // period))[:rows]), f"vector {b}"
        _, y64, ab = O.matvec(t, small, period, cols, X[0], threads=8)
        assert_dot_close(want[0], y64, ab, what="the repeated rows")
    finally:
        S.free()
        W.free()
