"""GPU: matvec launches whose last few tiles are split over workgroups.

With T tiles over G workgroups, the T mod G leftover tiles are cut into
ranges of X pairs (tile, stage).  Rows here leave one tile (16 rows past a
whole round of 256 workgroups, or one row past it), two, and a few dozen, so X is
an eighth of a tile, what one round of waves still takes, or the narrowest
width; the shares of a tile fill one batch of the exchange, two, or more.

Bar: rows within 2e-5 * sum|w*x| of the f64 dot, and the same bits on every
call (the counters and entries are handed back empty).
"""
import numpy as np
import pytest

import oracle_lib as O
import si_hip
from test_gpu_parity import assert_dot_close, log, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,rows,cols", [
    (12, 4112, 5120), (12, 4097, 12800), (12, 4128, 10240), (12, 4700, 7680), (12, 17408, 5120),
    (13, 4112, 10240), (13, 4113, 12544), (13, 8208, 6400),
    (14, 4112, 11264), (14, 4097, 14336), (14, 4608, 10240),
    (14, 8210, 5376), (14, 8224, 8448)])
def test_split_ranges(hip_ctx, t, rows, cols):
    log(f"split ranges t={t} {rows}x{cols}")
    w = si_hip.synth_matrix(t, seed=rows + 5 * cols, rows=rows, cols=cols, threads=8)
    x = si_hip.synth_normal(rows + cols + t, cols)
    _, y64, ab = O.matvec(t, w, rows, cols, x, threads=8)
    W = hip_ctx.upload_quant_weight_private(w, t)
    try:
        y = hip_ctx.gguf_quant_matvec_weight(W, rows, cols, x)
        assert_dot_close(y, y64, ab, what=f"{rows}x{cols}")
        for _ in range(3):
            assert same_bits(hip_ctx.gguf_quant_matvec_weight(W, rows, cols, x), y)
    finally:
        W.free()


@pytest.mark.parametrize("rows,cols", [(2816, 5120), (4352, 5120), (4112, 7680)])
def test_split_ranges_gate_up(hip_ctx, rows, cols):
    """Two matrices a tile (gate and up): fewer tiles than workgroups, and
    one and sixteen left over."""
    gw, uw = (si_hip.synth_matrix(12, seed=rows + k, rows=rows, cols=cols, threads=8)
              for k in (1, 2))
    x = si_hip.synth_normal(rows + cols, cols)
    (_, g, gb), (_, u, ub) = (O.matvec(12, w, rows, cols, x, threads=8) for w in (gw, uw))
    s = 1.0 / (1.0 + np.exp(np.minimum(-g, 700.0)))
    # |d silu / d g| <= 1.1; both dots within 2e-5 of their absolute sums
    bound = 2e-5 * (1.1 * gb * (np.abs(u) + 2e-5 * ub) + np.abs(g) * ub) + 1e-6 * np.abs(g * s * u)
    G, U = (hip_ctx.upload_quant_weight_private(w, 12) for w in (gw, uw))
    try:
        h = hip_ctx.q4_k_fused_gate_up_weights(G, U, rows, cols, x)
        assert np.all(np.abs(h - g * s * u) <= bound + 1e-30)
        assert same_bits(hip_ctx.q4_k_fused_gate_up_weights(G, U, rows, cols, x), h)
    finally:
        G.free()
        U.free()
