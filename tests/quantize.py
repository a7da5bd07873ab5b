"""Q4_K / Q5_K matrices quantised from given weights (test infrastructure).

Per 256-element block: each 32-element unit's least weight (at most 0) and its
step are written as 6-bit multiples of the block's halves d and dmin
(quant.rs:45-59, 107-121: weight = d sc q - dmin m).  On weights of zero mean the
two products are of one size everywhere and several times the weights.
"""
from __future__ import annotations

import numpy as np

from cancel_blocks import _scale_bytes


def quantize(t: int, w: np.ndarray) -> np.ndarray:
    """Packed blocks of the weights w (any shape, a multiple of 256), type 12 or 13."""
    top = 15 if t == 12 else 31
    u = np.asarray(w, np.float32).reshape(-1, 8, 32)
    n = u.shape[0]
    least = -np.minimum(u.min(2), 0.0)
    scale = (u.max(2) + least) / top
    d = (scale.max(1) / 63).astype(np.float16)
    dmin = (least.max(1) / 63).astype(np.float16)
    df, mf = (v.astype(np.float32)[:, None] for v in (d, dmin))
    sc = np.clip(np.rint(scale / df), 0, 63)
    mn = np.clip(np.rint(least / np.maximum(mf, 1e-12)), 0, 63)
    step = np.maximum(df * sc, 1e-12)[:, :, None]
    q = np.clip(np.rint((u + (mf * mn)[:, :, None]) / step), 0, top).astype(np.uint8)
    parts = [d.view(np.uint8).reshape(n, 2), dmin.view(np.uint8).reshape(n, 2),
             _scale_bytes(sc.astype(np.uint8), mn.astype(np.uint8))]
    if t == 13:
        parts.append(np.bitwise_or.reduce([(q[:, k] >> 4) << k for k in range(8)]))
    nib = q & 15
    parts.append((nib[:, 0::2] | (nib[:, 1::2] << 4)).reshape(n, 128))
    return np.ascontiguousarray(np.concatenate(parts, 1)).reshape(-1)


def terms(t: int, raw: np.ndarray):
    """Per block, the sums of d sc q and of dmin m over its weights, in f64."""
    b = raw.reshape(-1, 144 if t == 12 else 176)
    half = lambda at: b[:, at:at + 2].copy().view(np.float16).astype(np.float64)  # noqa: E731
    s = b[:, 4:16]
    sc = np.concatenate([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
    mn = np.concatenate([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
    qs = b[:, -128:].reshape(-1, 4, 1, 32)
    q = np.concatenate([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).astype(np.float64)
    if t == 13:
        q = q + 16 * ((b[:, None, 16:48] >> np.arange(8, dtype=np.uint8)[None, :, None]) & 1)
    return ((sc * q.sum(2)).sum(1) * half(0)[:, 0], 32 * mn.sum(1) * half(2)[:, 0])
