"""The same call gives the same bits every time: the products in every form, and a prompt through a hybrid stack."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SEED = 0xDA1A0025


@pytest.mark.parametrize("rows,cols,n", [
    (700, 1024, 2), (700, 1024, 4), (700, 1024, 8), (700, 1024, 16), (700, 1024, 60),  # few-column forms, blocks
    (200, 1024, 4100), (5120, 6144, 333),                                             # tiles, whole and split K
])
def test_products(dz, oracle, rows, cols, n):
    m = dz.Q1_0Matrix(oracle.synth_q1_0(SEED, 18, 0, rows, cols), rows, cols)
    x = np.random.default_rng(n).standard_normal((n, cols)).astype(np.float32)
    y = m.matvec_batch(x)
    for _ in range(10):
        assert np.array_equal(m.matvec_batch(x), y)


@pytest.mark.parametrize("n", [700, 16])
def test_forward(dz, n):
    cfg = dz.Config.bonsai27b(max_ctx=1024)
    cfg.n_layers, cfg.vocab = 4, 512
    ctx = dz.Context(dz.Model.synthetic(cfg, SEED))
    ids = np.random.default_rng(n).integers(0, cfg.vocab, n).astype(np.uint32)
    first = ctx.forward_batch(ids)
    for _ in range(6):
        ctx.reset()
        assert np.array_equal(ctx.forward_batch(ids), first)
