"""The n-token attention at the edges of its tiles, against the oracle: 64 (token, q-head) rows per
workgroup, position chunks of whole 16-position blocks, one chunk (gated output written by the kernel)
and several (merged), every GQA group size, chunks of one block and of many (from 32 blocks on the next block's
scores are formed ahead).

One attention layer over a random cache, so the batch's first token already sees `start` positions; bar:
1e-3 normwise, the repository's for logits, and 2e-5 against float64 attention's own rounding at these
lengths (about 500 f32 additions per output: 500 * 2^-24 = 3e-5 of the largest term, which a softmax's
convex sum does not reach).
"""
import numpy as np
import pytest

from conftest import normwise_rel

pytestmark = pytest.mark.gpu

SEED = 0xDA1A0021


@pytest.mark.parametrize("nq,nkv,start,n", [
    (2, 2, 0, 65),      # group 1: 65 rows, one past a tile; from an empty context
    (4, 2, 15, 33),     # group 2: 66 rows
    (3, 1, 16, 43),     # group 3: three tiles, the last of one row
    (4, 1, 300, 17),    # group 4: 68 rows, several chunks
    (6, 1, 47, 11),     # group 6: 66 rows
    (6, 1, 500, 10),    # group 6: 60 rows, one tile
    (8, 1, 129, 70),    # group 8
    (2, 1, 0, 1),       # a single token into an empty context
])
def test_tiles_and_chunks(dz, oracle, nq, nkv, start, n):
    cfg = dz.Config.small(n_layers=1, max_ctx=640, n_head=nq, n_head_kv=nkv, full_attn_interval=1, vocab=256)
    m, om = dz.Model.synthetic(cfg, SEED), oracle.Model(cfg, SEED)
    ctx = dz.Context(m)
    rng = np.random.default_rng(nq * 1000 + start + n)
    if start:
        k = rng.standard_normal((nkv, start, cfg.head_dim), dtype=np.float32) * 2
        v = rng.standard_normal((nkv, start, cfg.head_dim), dtype=np.float32)
        ctx.set_kv(0, k, v)
        om.set_kv(0, k, v)
        ctx.set_pos(start)
        om.set_pos(start)
    ids = rng.integers(0, cfg.vocab, n).astype(np.uint32)
    per = ctx.forward_batch(ids, per_pos_logits=True)
    for i, t in enumerate(ids):
        _, olg = om.forward(int(t))
        assert normwise_rel(per[i], olg) < 2e-5, i


def _chunks(nq, nkv, start, n):
    """bt_attn_mfma_chunks (model.hip): number of position chunks, positions of a chunk."""
    grp, ctx = nq // nkv, start + n
    wgs = -(-n * grp // 64) * nkv
    nch = 1 if wgs >= 256 else max(1, min(256, -(-(256 if n * grp <= 64 else 512) // wgs)))
    csz = -(-(-(-ctx // nch)) // 16) * 16
    return -(-ctx // csz), csz


@pytest.mark.parametrize("nq,nkv,start,n,nch,csz", [
    (8, 4, 1101, 1000, 4, 528),   # group 2: scores ahead, merged, every chunk and the last row tile ragged
    (16, 4, 30, 1021, 1, 1056),   # group 4: scores ahead, one chunk that ends 5 positions short of its blocks
    (40, 5, 20, 411, 1, 432),     # group 8: one chunk of 27 blocks
    (12, 2, 700, 300, 9, 112),    # group 6: nine chunks of seven blocks
])
def test_chunks_of_many_blocks(dz, oracle, nq, nkv, start, n, nch, csz):
    """Every token's output, through the keys and values that a second layer forms from it; the last one's logits.
    Bar as above."""
    assert _chunks(nq, nkv, start, n) == (nch, csz)
    cfg = dz.Config.small(n_layers=2, max_ctx=start + n, n_head=nq, n_head_kv=nkv, full_attn_interval=1, vocab=256)
    m, om = dz.Model.synthetic(cfg, SEED), oracle.Model(cfg, SEED)
    ctx = dz.Context(m)
    rng = np.random.default_rng(nq * 1000 + start + n)
    for layer in range(2):
        k = rng.standard_normal((nkv, start, cfg.head_dim), dtype=np.float32) * 2
        v = rng.standard_normal((nkv, start, cfg.head_dim), dtype=np.float32)
        ctx.set_kv(layer, k, v)
        om.set_kv(layer, k, v)
    ctx.set_pos(start)
    om.set_pos(start)
    ids = rng.integers(0, cfg.vocab, n).astype(np.uint32)
    last = ctx.forward_batch(ids)
    for t in ids:
        _, olg = om.forward(int(t))
    assert normwise_rel(last, olg) < 2e-5
    for layer in range(2):
        kg, vg = ctx.get_kv(layer, start + n)
        ko, vo = om.get_kv(layer)
        for a, b in ((kg, ko), (vg, vo)):
            a, b = a[:, start:].astype(np.float64), b[:, start:].astype(np.float64)
            err = np.abs(a - b).max(axis=(0, 2)) / np.abs(b).max(axis=(0, 2))
            assert err.max() < 2e-5, (layer, int(err.argmax()), err.max())
