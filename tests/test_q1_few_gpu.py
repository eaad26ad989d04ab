"""The few-column Q1_0 product (n <= 16) in each of its forms (2, 4, 8 and 16 tokens per operand) at the edges of
its tiles, against float64; and the forward that hands its activations over as digits (up to 16 tokens) against
the oracle.

Bound of the product: the sums of a group's digits and of the groups are f32 additions of partial sums, at most
(8 + 2 ngroups) per slot (two fmas join a group's sums in the forms of four and eight tokens) and 8 between the
slots and splits, and the digits keep 2^-29 (n <= 4: 2^-39) of their 32-column block's largest value:
|err| <= (2 ngroups + 24) 2^-24 Σ|w x| + 2^-29 Σ|w| max|x|.
"""
import numpy as np
import pytest

from conftest import normwise_rel

pytestmark = pytest.mark.gpu

SEED = 0xDA1A0023


def _matrix(rng, rows, cols):
    blk = np.empty((rows, cols // 128, 18), np.uint8)
    blk[:, :, 2:] = rng.integers(0, 256, (rows, cols // 128, 16), dtype=np.uint8)
    sc = (np.abs(rng.standard_normal((rows, cols // 128))) * 0.02).astype(np.float16)
    blk[:, :, :2] = sc[..., None].view(np.uint8)
    sign = np.unpackbits(blk[:, :, 2:], axis=-1, bitorder="little").astype(np.float64) * 2 - 1
    return blk.reshape(-1), (sign * sc[..., None].astype(np.float64)).reshape(rows, cols)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("rows,cols", [(1, 128), (65, 640), (511, 1152), (2100, 512), (70, 17408),  # two waves a row-block
                                       (66100, 256)])  # a wave each (more than half of the CUs have a workgroup)
def test_forms(dz, n, rows, cols):
    rng = np.random.default_rng(rows * 31 + cols + n)
    aos, w = _matrix(rng, rows, cols)
    m = dz.Q1_0Matrix(aos, rows, cols)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    x[:, ::97] *= np.float32(2.0 ** 12)
    x[0, :32] = 0
    y0 = rng.standard_normal((n, rows)).astype(np.float32)
    ref = x.astype(np.float64) @ w.T
    bound = ((2 * (cols // 128) + 24) * 2.0 ** -24 * (np.abs(x.astype(np.float64)) @ np.abs(w).T)
             + 2.0 ** -29 * np.abs(x).max(1)[:, None] * np.abs(w).sum(1)[None])
    y = m.matvec_batch(x)
    assert np.all(np.abs(y - ref) <= bound)
    ya = y0.copy()
    m.matvec_add_batch_into_slice(x, n, ya)
    assert np.all(np.abs(ya - (y0 + ref)) <= bound + 2.0 ** -23 * (np.abs(y0) + np.abs(ya)))


@pytest.mark.parametrize("n", [1, 2, 3, 4])
def test_small_values_beside_large_ones(dz, n):
    """Up to four columns, an f32 ten powers of two below the largest of its block comes through with every bit:
    two values 2^10 that cancel in the row, and one with its lowest significand bits set beside them."""
    rows, cols = 64, 256
    rng = np.random.default_rng(n)
    blk = np.empty((rows, cols // 128, 18), np.uint8)
    blk[:, :, 2:] = rng.integers(0, 256, (rows, cols // 128, 16), dtype=np.uint8)
    blk[:, :, 0], blk[:, :, 1] = 0x00, 0x3C  # f16 1.0
    blk[:, :, 2] = blk[:, :, 2] & 0xFC | 1   # column 0 of a group is +, column 1 is -
    m = dz.Q1_0Matrix(blk.reshape(-1), rows, cols)
    v = (1 + (rng.integers(0, 1 << 23, n) | 3) / 2.0 ** 23).astype(np.float32)
    x = np.zeros((n, cols), np.float32)
    x[:, 128] = x[:, 129] = 2.0 ** 10
    x[:, 128 + 21] = v
    sign = ((blk[:, 1, 2 + 21 // 8] >> (21 % 8)) & 1).astype(np.float32) * 2 - 1
    assert np.array_equal(m.matvec_batch(x), sign[None] * v[:, None])


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8])
def test_large_values_that_cancel(dz, n):
    """Two values of 2^20 and more that cancel in every group of every row, among standard normal ones: up to eight
    columns the sums of the largest digits round nothing else away, so the error is that of the digits' grid, at most
    2^-29 (n <= 4: 2^-39) of the large value per column against results of columns of size 1, and f32 rounding."""
    rows, cols = 512, 2048
    rng = np.random.default_rng(n)
    aos, _ = _matrix(rng, rows, cols)
    blk = aos.reshape(rows, cols // 128, 18)
    blk[:, :, 2 + 5] = (blk[:, :, 2 + 5] & 0xFE) | (1 - ((blk[:, :, 2] >> 3) & 1))  # column 40's sign: not column 3's
    sign = np.unpackbits(blk[:, :, 2:], axis=-1, bitorder="little").astype(np.float64) * 2 - 1
    w = (sign * np.ascontiguousarray(blk[:, :, :2]).view(np.float16).astype(np.float64)).reshape(rows, cols)
    m = dz.Q1_0Matrix(np.ascontiguousarray(blk.reshape(-1)), rows, cols)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    x[:, 3::128] = x[:, 40::128] = 2.0 ** 20 * (1 + rng.random((n, cols // 128)))
    ref = x.astype(np.float64) @ w.T
    err = np.linalg.norm(m.matvec_batch(x) - ref) / np.linalg.norm(ref)
    assert err < 2.0 ** 21 * 2.0 ** (-39 if n <= 4 else -29) + 1e-6, err


def test_non_finite_token(dz):
    rng = np.random.default_rng(9)
    aos, _ = _matrix(rng, 130, 1024)
    m = dz.Q1_0Matrix(aos, 130, 1024)
    for n in (2, 4, 8, 16):
        x = rng.standard_normal((n, 1024)).astype(np.float32)
        good = m.matvec_batch(x)
        bad = x.copy()
        bad[n - 1, 700] = -np.inf
        y = m.matvec_batch(bad)
        assert np.all(np.isnan(y[n - 1])) and np.array_equal(y[:n - 1], good[:n - 1])


@pytest.mark.parametrize("n", [1, 2, 3, 5, 9, 16])
def test_short_batches(dz, oracle, n):
    """hidden and FFN widths that end inside a K tile (640 and 896 columns), nine v-heads (a tile of one head)."""
    cfg = dz.Config.small(n_layers=4, max_ctx=64, hidden=640, ffn=896, vocab=300, ssm_k_heads=1, ssm_v_heads=9)
    m, om = dz.Model.synthetic(cfg, SEED), oracle.Model(cfg, SEED)
    ctx = dz.Context(m)
    rng = np.random.default_rng(n)
    for _ in range(2):
        ids = rng.integers(0, cfg.vocab, n).astype(np.uint32)
        logits = ctx.verify_forward(ids)
        ctx.verify_commit(n)
        for i, t in enumerate(ids):
            _, olg = om.forward(int(t))
            assert normwise_rel(logits[i], olg) < 2e-5, i  # four layers of f32 sums, about 1e-6 each
    ids = rng.integers(0, cfg.vocab, n).astype(np.uint32)
    last = ctx.forward_batch(ids)
    for t in ids:
        _, olg = om.forward(int(t))
    assert normwise_rel(last, olg) < 2e-5
