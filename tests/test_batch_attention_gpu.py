"""The n-token attention at the edges of its tiles, against the oracle: 64 (token, q-head) rows per
workgroup, position chunks of whole 16-position blocks, one chunk (gated output written by the kernel)
and several (merged), every GQA group size.

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
