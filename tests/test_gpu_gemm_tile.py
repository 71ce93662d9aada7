"""Quantised weights times several f32 vectors on the bf16 matrix cores
(gemm_tile.hip; qmm.matMulQ8_0's role, qmm.zig:58-138), at the edges of its
tiles, against the float64 product of the reference's dequantised weights
(dequant.zig:316-390).

Bound: a vector element enters as two bf16 numbers, off by at most 2^-17 of
itself; the f32 sums (products of 32 columns, then the blocks of a wave, then
the waves) round at most cols + 16 times, 2^-24 of the running sum each,
together at most (cols + 16) 2^-24 sum |w x|.
"""
import numpy as np
import pytest

import mmhip as mm

pytestmark = pytest.mark.gpu


def _check(y, x, w):
    exact = x.astype(np.float64) @ w.T
    bound = (2.0 ** -17 + (x.shape[1] + 16) * 2.0 ** -24) * (np.abs(x.astype(np.float64)) @ np.abs(w).T)
    err = np.abs(y.astype(np.float64) - exact)
    print(f"error / bound at most {float((err / np.maximum(bound, 1e-300)).max()):.3f}")
    assert np.all(err <= bound)


# One case at least per tile shape (256 CUs: 16x32, 16x64, 32x64 by eight
# waves, 32x64 by four), with ragged rows, vectors, columns and row groups.
@pytest.mark.parametrize("fmt,rows,cols,batch,layout", [
    (mm.Q8_0, 33, 2080, 2, 0), (mm.Q8_0, 300, 2592, 17, 1), (mm.Q8_0, 4100, 2080, 47, 0),
    (mm.Q8_0, 4000, 2080, 99, 0), (mm.Q8_0, 4100, 96, 129, 1), (mm.Q8_0, 4100, 32, 256, 0),
    (mm.IQ2_XXS, 33, 256, 2, 0), (mm.IQ2_XXS, 17, 768, 16, 1), (mm.IQ2_XXS, 4100, 2304, 47, 0),
    (mm.IQ2_XXS, 4000, 512, 99, 0), (mm.IQ2_XXS, 4100, 256, 129, 1), (mm.IQ2_XXS, 8, 1280, 33, 0)])
def test_tile_edges(ctx, orc, fmt, rows, cols, batch, layout):
    rng = np.random.default_rng(rows * 7 + cols + batch)
    raw = mm.make_weight(rng, fmt, rows, cols)
    w = orc.dequantize(raw, fmt, rows * cols).reshape(rows, cols).astype(np.float64)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    x[0] *= 1e-20
    x[batch - 1, :: 5] *= 1e4
    wt = ctx.upload(raw, fmt, rows, cols)
    dx, dy = mm.DeviceArray.from_numpy(ctx, x), mm.DeviceArray(ctx, 4 * batch * rows)
    ctx.qmm_dev(wt, 0, dx, dy, batch, layout)
    ctx.synchronize()
    y = dy.to_numpy(np.float32, batch * rows)
    for h in (wt, dx, dy):
        h.free()
    y = y.reshape(batch, rows) if layout == 0 else y.reshape(rows, batch).T
    _check(y, x, w)


@pytest.mark.parametrize("fmt", [mm.Q8_0, mm.IQ2_XXS])
def test_extreme_vectors(ctx, orc, fmt):
    """Vectors up to f32's largest, whose products with the integer weights
    pass it before the block scale brings them back; an infinity and a NaN
    poison their own vector only."""
    rng = np.random.default_rng(77 + fmt)
    rows, cols, batch = 40, 2304, 5
    raw = mm.make_weight(rng, fmt, rows, cols)
    w = orc.dequantize(raw, fmt, rows * cols).reshape(rows, cols).astype(np.float64)
    w_sum = np.abs(w).sum(axis=1).max()
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    x[0] = np.float32(3.0e38 / max(w_sum, 1.0)) * rng.choice([-1.0, 1.0], cols).astype(np.float32)
    x[1, 7], x[3, cols - 1] = np.inf, np.nan
    y = ctx.batch_mat_mul(raw, fmt, x, rows, batch, cols)
    _check(y[[0, 2, 4]], x[[0, 2, 4]], w)
    assert np.all(np.isnan(y[[1, 3]]))


@pytest.mark.parametrize("exp", [-104, -112, -120])
@pytest.mark.parametrize("fmt", [mm.Q8_0, mm.IQ2_XXS])
def test_tiny_vectors(ctx, orc, fmt, exp):
    """Below 2^-105 an element's second part is a subnormal bf16 number: off by at
    most 2^-134, which the 2^-12 that vectors enter with makes 2^-122."""
    rng = np.random.default_rng(79 + fmt - exp)
    rows, cols, batch = 40, 2304, 5
    raw = mm.make_weight(rng, fmt, rows, cols)
    w = orc.dequantize(raw, fmt, rows * cols).reshape(rows, cols).astype(np.float64)
    x = np.ldexp(rng.uniform(0.5, 1.0, (batch, cols)) * rng.choice([-1.0, 1.0], (batch, cols)), exp).astype(np.float32)
    y = ctx.batch_mat_mul(raw, fmt, x, rows, batch, cols)
    x64 = x.astype(np.float64)
    err = np.abs(y.astype(np.float64) - x64 @ w.T)
    off = np.maximum(2.0 ** -17 * np.abs(x64), 2.0 ** -122)
    # The f32 sums as in the bound above, and half a smallest f32 per output block.
    bound = (off + (cols + 16) * 2.0 ** -24 * np.abs(x64)) @ np.abs(w).T + cols * 2.0 ** -149
    print(f"error / bound at most {float((err / bound).max()):.3f}")
    assert np.all(err <= bound)


def test_infinite_block_scale(ctx, orc):
    """IQ2_XXS superblocks of infinite scale, sub-block scale codes of zero among
    them, times vectors of the weights' signs: every product is +inf, and so is
    the sum (the CPU path's result, dequant.zig:316-355)."""
    rng = np.random.default_rng(78)
    rows, cols = 16, 768
    raw = mm.make_iq2_xxs(rng, rows, cols).reshape(rows, cols // 256, 66)
    raw[:, :, :2] = np.array([0x3C00], np.uint16).view(np.uint8)  # 1.0
    signs = np.sign(orc.dequantize(raw.reshape(-1), mm.IQ2_XXS, rows * cols)).reshape(rows, cols).astype(np.float32)
    raw[:, 1, :2] = np.array([0x7C00], np.uint16).view(np.uint8)  # inf
    y = ctx.batch_mat_mul(raw.reshape(-1), mm.IQ2_XXS, signs, rows, rows, cols)
    assert np.all(np.diagonal(y) == np.inf)
