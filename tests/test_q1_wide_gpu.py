"""The many-token Q1_0 product at the edges of its tiles: 512-row and 32-token workgroup tiles, 16-row and 16-token
operand blocks, half and whole K tiles, split and unsplit K.  More than 16 columns go to it past a line in (64-row
block, K tile, 16 columns) units, below it in blocks of 16 to the few-column form; every case names its side.

Bound: with u = 2^-24, a group of 128 columns takes six f32 additions and one fma into the row's sum, and
the activations' digits keep 2^-29 of their 32-column block's largest value, so a row's error is at most
(ngroups + 8) u Σ|w x| + 2^-29 Σ|w| max|x|, which the comparison below uses as it stands (the accumulate
form and the split sums add one rounding each).
"""
import os
import re

import numpy as np
import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu


def is_wide(rows, cols, n):
    """Whether matvec_batch takes the tiles (few_blocks in q1_mat.hip, from the source's own constant)."""
    with open(os.path.join(ROOT, "daiza_amd", "csrc", "q1_mat.hip")) as f:
        line = int(re.search(r"constexpr int kFewWaves = (\d+);", f.read()).group(1))
    return n > 16 and -(-rows // 64) * -(-cols // 512) * -(-n // 16) > line


def _matrix(rng, rows, cols):
    blk = np.empty((rows, cols // 128, 18), np.uint8)
    blk[:, :, 2:] = rng.integers(0, 256, (rows, cols // 128, 16), dtype=np.uint8)
    sc = (np.abs(rng.standard_normal((rows, cols // 128))) * 0.02).astype(np.float16)
    blk[:, :, :2] = sc[..., None].view(np.uint8)
    sign = np.unpackbits(blk[:, :, 2:], axis=-1, bitorder="little").astype(np.float64) * 2 - 1
    return blk.reshape(-1), (sign * sc[..., None].astype(np.float64)).reshape(rows, cols)


def _check(y, w, x, extra=0.0):
    ref = x.astype(np.float64) @ w.T
    u = 2.0 ** -24
    mass = np.abs(x.astype(np.float64)) @ np.abs(w).T
    bound = (w.shape[1] // 128 + 8 + 8) * u * mass + 2.0 ** -29 * np.abs(x).max(1)[:, None] * np.abs(w).sum(1)[None]
    err = np.abs(y - ref)
    assert np.all(err <= bound + extra), float((err / (bound + extra)).max())


@pytest.mark.parametrize("rows,cols,n", [
    (1, 128, 1024 * 32 + 17),   # one row, one group of the first half tile, half a token group and one
    (16, 256, 1025 * 32),       # one operand block, a whole half tile, whole token groups
    (511, 384, 129 * 32 + 1),   # a row short of a tile, three groups, one token into the last token group
    (513, 640, 57 * 32 + 31),   # one row into the second row group, one group into the second tile
    (1088, 1152, 20 * 32 + 16),  # three row groups, half a token group
    (8 * 64 * 9 + 5, 512, 14 * 32 + 16),  # more than one band of row groups
    (5120, 17408, 40),          # few workgroups: K is split
    (200, 17408, 250),          # the same with half of a row group
])
def test_tile_edges(dz, rows, cols, n):
    assert is_wide(rows, cols, n)
    rng = np.random.default_rng(rows + cols + n)
    aos, w = _matrix(rng, rows, cols)
    m = dz.Q1_0Matrix(aos, rows, cols)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    _check(m.matvec_batch(x), w, x)
    y0 = rng.standard_normal((n, rows)).astype(np.float32)
    y = y0.copy()
    m.matvec_add_batch_into_slice(x, n, y)
    _check(y - y0.astype(np.float64), w, x, extra=2.0 ** -23 * (np.abs(y0) + np.abs(y)))


@pytest.mark.parametrize("n", [20, 4100])
def test_block_ranges_and_non_finite(dz, n):
    """Blocks of 32 columns of very different size, tiny and huge values; a token with an infinity or a
    NaN gives NaN in its own results and leaves the others as they are."""
    rows, cols = 200, 1024
    assert is_wide(rows, cols, n) == (n > 20)
    rng = np.random.default_rng(3)
    aos, w = _matrix(rng, rows, cols)
    m = dz.Q1_0Matrix(aos, rows, cols)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    x[0, 32:64] *= np.float32(2.0 ** 30)
    x[1, ::32] *= np.float32(2.0 ** -20)
    x[2] *= np.float32(2.0 ** -90)
    x[3] *= np.float32(2.0 ** 100)
    x[4] = 0
    x[5, 64:] = 0
    y = m.matvec_batch(x)
    _check(y, w, x)
    assert np.all(y[4] == 0)
    bad = x.copy()
    bad[7, 500], bad[9, 0] = np.inf, np.nan
    yb = m.matvec_batch(bad)
    assert np.all(np.isnan(yb[7])) and np.all(np.isnan(yb[9]))
    keep = [i for i in range(n) if i not in (7, 9)]
    assert np.array_equal(yb[keep], y[keep])


@pytest.mark.parametrize("n", [1, 2, 4, 7, 16, 20, 8225])
def test_ends_of_the_range(dz, n):
    """Activations near the ends of f32's exponent range, in every form of the product: tiny ones keep their
    precision, and a group's terms do not overflow where the f16 scale brings the result back."""
    rows, cols = 96, 640
    assert is_wide(rows, cols, n) == (n > 20)
    rng = np.random.default_rng(n)
    aos, w = _matrix(rng, rows, cols)
    m = dz.Q1_0Matrix(aos, rows, cols)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    for e in (-100, -93, -86, 110, 120):
        xe = np.ldexp(x, e)
        _check(m.matvec_batch(xe), w, xe)
    # one group whose 128 terms of 2^122 have one sign in row 0: 2^129 before the scale, and every row's
    # result at most 2^129 max(scale), which is finite
    big = np.zeros_like(x)
    big[:, :128] = np.ldexp(np.sign(w[0, :128]), 122)
    assert 2.0 ** 129 * np.abs(w[:, :128]).max() < 2.0 ** 127
    _check(m.matvec_batch(big), w, big)


@pytest.mark.parametrize("rows,cols,n,wide", [
    (4613, 1152, 161, True),   # above the line between the 16-column blocks and the 512 x 32 tiles: ragged rows, half a
    (5121, 640, 207, True),    # K tile, a token past a tile; one row into the last row group
    (8192, 512, 256, False),   # the line itself (2048 units): blocks
    (8192, 512, 257, True),    # and one column past it: tiles
    (130, 1664, 250, False),   # blocks: three row-blocks, a ragged last block of columns, split K
])
def test_both_sides_of_the_block_line(dz, rows, cols, n, wide):
    assert is_wide(rows, cols, n) == wide
    rng = np.random.default_rng(rows + n)
    aos, w = _matrix(rng, rows, cols)
    m = dz.Q1_0Matrix(aos, rows, cols)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    _check(m.matvec_batch(x), w, x)
    y0 = rng.standard_normal((n, rows)).astype(np.float32)
    y = y0.copy()
    m.matvec_add_batch_into_slice(x, n, y)
    _check(y - y0.astype(np.float64), w, x, extra=2.0 ** -23 * (np.abs(y0) + np.abs(y)))
