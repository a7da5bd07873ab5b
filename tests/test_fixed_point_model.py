"""CPU model of the matrix-core kernels' activation handling (no GPU).

The kernels (memory-aware-inference_amd/csrc/mfma_common.h, tokens_common.h)
write each 256-element block of x as X * 2^(e - 30), X an integer of at most 30
bits and e the exponent of the block's largest |x| (largest |x| < 2^e).
Non-zero activations below 2^(e - 14) are "side" elements: they stay in X,
rounded like the rest, and the kernels count them, half a unit 2^(e - 31) each.

  * "one": the kernels of one and two vectors.  Per row and stage (four or two
    blocks) the bound (largest |w| of a 64-element share) x (half units of the
    share's side elements) is compared with the sum of the shares' |partial
    dot|: a row where it exceeds 4e-6 of that recomputes exactly.
  * "rows": the kernels with two to sixteen vectors in the matrix-core rows.  Per
    row and slice of at most four blocks the bound (largest |w| of the slice) x
    (half units of a block's side elements) may be 2^-21 of the sum of |block
    dot| for blocks of at most eight side elements and 4e-6 for the others; a
    slice past that is recomputed exactly.

A block with a non-finite or huge activation takes the exact path.  This model
restates those rules in numpy and measures the error they leave against the f64
dot.  (The kernels bound |w| by what a block's header allows, the model by the
weights themselves, so it lets more pass.)  Elements kept in X have a relative
error of at most 2^-17, and the side elements cost at most 4e-6 of sum|w*x|, so
the activation rounding stays below (2^-17 + 4e-6) * sum|w*x|, 0.58 of the 2e-5
bar, whatever the weights.  The rule the kernels used before (a block goes exact
only when a whole 16-element chunk lies 2^13 below the block maximum) is modelled
too, to show that the crafted input does catch it.
"""
import numpy as np
import pytest

import crafted
import oracle_lib as O
import si_hip

BAR = 2e-5
SIDE_SHIFT = 14
FEW, FEW_TOL = 8, 2.0 ** -21
TOL = 4e-6
LIMIT = (2.0 ** -17 + TOL) / BAR  # 0.58
KERNELS = [("one", 4), ("one", 2), ("rows", 4)]


def _block_split(v):
    """(kind, fixed-point x, half units of its side elements) of one block, kind in
    fixed/rounded/exact."""
    a = np.abs(v)
    none = np.zeros(v.shape)
    if not (np.all(np.isfinite(v)) and np.all(a < 2.0 ** 100)):
        return "exact", v, none
    e = int(np.frexp(float(a.max()))[1])  # largest |x| < 2^e
    fixed = np.rint(np.ldexp(v, 30 - e)) * 2.0 ** (e - 30)
    side = (v != 0) & (a < 2.0 ** (e - SIDE_SHIFT))
    return ("rounded" if side.any() else "fixed"), fixed, side * 2.0 ** (e - 31)


def _slices(nb, kernel, stage):
    """[first, end) of the stages, or of the slices (one block at the end takes
    another from the slice before it)."""
    first = list(range(0, nb, stage)) + [nb]
    if kernel == "rows" and len(first) > 2 and first[-1] - first[-2] == 1:
        first[-2] -= 1
    return list(zip(first, first[1:]))


def model_dot(w, x, rule="side", kernel="one", stage=4):
    """The kernel's activation handling for every row of w: returns
    (y as the kernel would compute it in exact arithmetic, per-block kinds,
    number of row-stages that are recomputed exactly)."""
    x64 = np.asarray(x, np.float32).astype(np.float64)
    nb = x64.size // 256
    xb = x64.reshape(nb, 256)
    kinds, xe, half = [], np.empty_like(xb), np.zeros_like(xb)
    for b in range(nb):
        if rule == "side":
            k, f, half[b] = _block_split(xb[b])
        else:  # the chunk rule
            v = xb[b]
            a = np.abs(v)
            amax = float(a.max())
            e = int(np.frexp(amax)[1])
            cmax = a.reshape(16, 16).max(axis=1)
            bad = not np.all(np.isfinite(v)) or np.any((cmax > 0) & (cmax < amax * 2.0 ** -13))
            k, f = ("exact", v) if bad else ("fixed", np.rint(np.ldexp(v, 30 - e)) * 2.0 ** (e - 30))
        kinds.append(k)
        xe[b] = f
    rows = w.shape[0]
    wb = w.reshape(rows, nb, 256)
    # per row, block and 64-element share: the dot with the kernel's x
    shares = np.einsum("rbgk,bgk->rbg", wb.reshape(rows, nb, 4, 64), xe.reshape(nb, 4, 64))
    y = shares.sum(axis=(1, 2))
    redone = 0
    for s0, s1 in _slices(nb, kernel, stage):
        blocks = [b for b in range(s0, s1) if kinds[b] == "rounded"]
        if not blocks:
            continue
        err = np.zeros(rows)  # over the tolerance
        for b in blocks:
            if kernel == "one":
                wmax = np.abs(wb[:, b, :]).reshape(rows, 4, 64).max(axis=2)
                err += (wmax * half[b].reshape(4, 64).sum(axis=1)).sum(axis=1) / TOL
            else:
                tol = FEW_TOL if np.count_nonzero(half[b]) <= FEW else TOL
                err += np.abs(wb[:, s0:s1]).max(axis=(1, 2)) * half[b].sum() / tol
        part = shares[:, s0:s1]
        a = np.abs(part).sum(axis=(1, 2)) if kernel == "one" else np.abs(part.sum(2)).sum(1)
        fail = ~(err * 1.02 <= a)
        redone += int(fail.sum())
        for b in blocks:  # the failing rows' rounded blocks, exactly
            y[fail] += wb[fail, b, :] @ (xb[b] - xe[b])
    return y, kinds, redone


def error_ratio(w, x, rule="side", kernel="one", stage=4):
    y, _, _ = model_dot(w, x, rule, kernel, stage)
    x64 = np.asarray(x, np.float32).astype(np.float64)
    err = np.abs(y - w @ x64)
    return float(np.max(err / (BAR * (np.abs(w) @ np.abs(x64)))))


def _weights(t, rows, cols, seed):
    raw = crafted.zero_weight_matrix(t, rows, cols, seed)
    w = O.dequantize(t, raw, rows * cols).reshape(rows, cols).astype(np.float64)
    assert np.all(w.reshape(rows, -1, 256)[:, :, crafted.ZERO_ELEMS] == 0.0)
    return w


@pytest.mark.parametrize("t", [12, 13, 14])
def test_crafted_weights_are_zero_where_asked(t):
    _weights(t, 8, 1024, 5 + t)


@pytest.mark.parametrize("kernel,stage", KERNELS)
@pytest.mark.parametrize("t", [12, 13, 14])
@pytest.mark.parametrize("case", crafted.CASES)
def test_side_rule_meets_the_bar_on_crafted_inputs(t, case, kernel, stage):
    rows, cols = 24, 2048
    w = _weights(t, rows, cols, 40 + t)
    x = crafted.crafted_x(cols, case, 7 + t)
    ratio = error_ratio(w, x, kernel=kernel, stage=stage)
    assert ratio <= LIMIT, f"{case}: {ratio:.3g} of the bar"
    if case == "side" and kernel == "rows":  # its other activations are exact
        assert ratio <= FEW_TOL / BAR


@pytest.mark.parametrize("kernel,tol", [("one", TOL), ("rows", FEW_TOL)])
@pytest.mark.parametrize("t", [12, 13, 14])
@pytest.mark.parametrize("nb", [4, 9])
def test_dot_that_side_elements_carry(t, nb, kernel, tol):
    """Eight side elements a block, each off by half a unit, 2^-17 of itself."""
    raw, x = crafted.small_dot(t, 3, 256 * nb)
    w = O.dequantize(t, raw, 3 * 256 * nb).reshape(3, -1).astype(np.float64)
    assert error_ratio(w, x, kernel=kernel) <= tol / BAR


def test_chunk_rule_fails_the_crafted_input():
    """The crafted "tiny" input is the case the chunk rule let through."""
    w = _weights(14, 24, 2048, 77)
    x = crafted.crafted_x(2048, "tiny", 78)
    assert error_ratio(w, x, "chunk") > 10.0
    assert error_ratio(w, x) <= LIMIT


def test_crafted_tiny_blocks_are_rounded_and_redone():
    """All small activations on the weights: every rounded block fails the
    check (its error bound is large against its own dot) and is redone."""
    w = _weights(12, 16, 1024, 3)
    y, kinds, redone = model_dot(w, crafted.crafted_x(1024, "tiny", 3))
    assert kinds == ["rounded"] * 4
    assert redone == 16


def test_crafted_many_blocks_are_rounded_and_pass():
    w = _weights(13, 16, 2048, 4)
    y, kinds, redone = model_dot(w, crafted.crafted_x(2048, "many", 4))
    assert kinds == ["rounded"] * 8
    assert redone == 0


def test_side_rule_routes_crafted_blocks():
    w = np.ones((2, 9 * 256))
    x = crafted.crafted_x(9 * 256, "side", 3)
    for kernel, stage in KERNELS:
        _, kinds, redone = model_dot(w, x, kernel=kernel, stage=stage)
        assert kinds == ["rounded"] * 9  # 1..8 side elements per block
        assert redone == 0
    _, kinds, _ = model_dot(w[:, :512], crafted.crafted_x(2 * 256, "edge", 3))
    assert kinds == ["fixed", "fixed"]


def test_slices():
    assert _slices(1, "rows", 4) == [(0, 1)]
    assert _slices(5, "rows", 4) == [(0, 3), (3, 5)]
    assert _slices(9, "rows", 4) == [(0, 4), (4, 7), (7, 9)]
    assert _slices(6, "rows", 4) == [(0, 4), (4, 6)]


def test_side_elements_are_rare_on_normal_activations():
    """Share of N(0,1) blocks with side elements, over 20,000 blocks, and with more
    than eight; the rows pass the checks on random weights."""
    x = si_hip.synth_normal(12345, 20000 * 256)
    blocks = x.astype(np.float64).reshape(-1, 256)
    split = [_block_split(v) for v in blocks]
    side = np.mean([k == "rounded" for k, _, _ in split])
    many = np.mean([np.count_nonzero(h) > FEW for _, _, h in split])
    print(f"N(0,1) blocks: {side:.4f} with side elements, {many:.6f} with more than {FEW}")
    assert 0.0 < side < 0.1
    assert many < 1e-4
    raw = si_hip.synth_matrix(12, seed=11, rows=64, cols=64 * 256)
    w = O.dequantize(12, raw, 64 * 64 * 256).reshape(64, -1).astype(np.float64)
    for kernel, stage in KERNELS:
        _, kinds, redone = model_dot(w, x[:64 * 256], kernel=kernel, stage=stage)
        assert "rounded" in kinds and redone == 0


def test_swiglu_intermediate_is_rounded_not_redone():
    """h = silu(g) * u of large random projections: half of h is many orders
    of magnitude below the block maximum, so every block is rounded; the
    check passes on the rows (the bound is tiny against the dot)."""
    rng = np.random.default_rng(9)
    g = rng.normal(0, 35, 4096)
    u = rng.normal(0, 35, 4096)
    h = (g / (1 + np.exp(-g)) * u).astype(np.float32)
    raw = si_hip.synth_matrix(14, seed=10, rows=64, cols=4096)
    w = O.dequantize(14, raw, 64 * 4096).reshape(64, 4096).astype(np.float64)
    y, kinds, redone = model_dot(w, h)
    assert kinds.count("rounded") >= 14
    assert redone == 0
    assert error_ratio(w, h) <= LIMIT


@pytest.mark.parametrize("kernel", ["one", "rows"])
@pytest.mark.parametrize("seed", range(3))
def test_side_rule_on_heavy_tailed_activations(seed, kernel):
    """Student-t activations with a few massive channels (the shape of real
    decoder activations) on random Q4_K weights."""
    rows, cols = 32, 4096
    raw = si_hip.synth_matrix(12, seed=seed, rows=rows, cols=cols)
    w = O.dequantize(12, raw, rows * cols).reshape(rows, cols).astype(np.float64)
    rng = np.random.default_rng(seed)
    x = rng.standard_t(2.0, cols)
    x[rng.choice(cols, 6, replace=False)] *= 1e4
    assert error_ratio(w, x.astype(np.float32), kernel=kernel) <= LIMIT
