"""The chunked delta rule of a prefill (33 tokens and more, 32 at a time) at the edges of its chunks, and the
token-by-token kernel below it, against the oracle: logits, DeltaNet states and conv rings from a seeded
state.

Bar: 1e-3 normwise, the repository's for logits and states, and here 2e-5: a state sums at most 130 f32
terms per element in either order (130 * 2^-24 = 8e-6 of the largest term) and the layer's products add
about 1e-6.
"""
import numpy as np
import pytest

from conftest import normwise_rel
from named_tensors import named_tensors

pytestmark = pytest.mark.gpu

SEED = 0xDA1A0022


@pytest.mark.parametrize("n", [32, 33, 63, 64, 65, 96, 130])
@pytest.mark.parametrize("nkh,nvh", [(2, 6), (1, 9)])
def test_chunk_edges(dz, oracle, n, nkh, nvh):
    cfg = dz.Config.small(n_layers=1, max_ctx=160, vocab=256, ssm_k_heads=nkh, ssm_v_heads=nvh)
    m, om = dz.Model.synthetic(cfg, SEED), oracle.Model(cfg, SEED)
    ctx = dz.Context(m)
    rng = np.random.default_rng(n + nvh)
    st = (rng.standard_normal((nvh, 128, 128)) * 0.1).astype(np.float32)
    conv = (rng.standard_normal((4, cfg.qkv_dim)) * 0.3).astype(np.float32)
    ctx.set_ssm_state(0, st, conv, 2)
    om.set_ssm_state(0, st, conv, 2)
    ids = rng.integers(0, cfg.vocab, n).astype(np.uint32)
    ids[5:12] = ids[4]  # repeated tokens: nearly parallel keys
    per = ctx.forward_batch(ids, per_pos_logits=True)
    for i, t in enumerate(ids):
        _, olg = om.forward(int(t))
        assert normwise_rel(per[i], olg) < 2e-5, i
    sg, cg, hg = ctx.get_ssm_state(0)
    so, co, ho = om.get_ssm_state(0)
    assert hg == ho and normwise_rel(sg, so) < 2e-5 and normwise_rel(cg, co) < 2e-5


def test_decay_that_clears_the_state(dz, oracle):
    """Gates whose decay underflows to 0 (ln a down to -inf) in some heads: a chunk's tokens behind such a token,
    and the final state, as the token-by-token kernel (32 tokens at a time) has them."""
    cfg = dz.Config.small(n_layers=1, max_ctx=160, vocab=256, ssm_k_heads=2, ssm_v_heads=6)
    om = oracle.Model(cfg, SEED)
    t = named_tensors(oracle, om, cfg, SEED)
    kind, a = t["blk.0.ssm_a"]
    a = a.copy()
    a[:4] = [-3e38, -1e30, -200.0, -1e5]
    t["blk.0.ssm_a"] = (kind, a)
    kind, dt = t["blk.0.ssm_dt.bias"]
    dt = dt.copy()
    dt[0] = 30.0  # softplus 30: ln a is -inf
    t["blk.0.ssm_dt.bias"] = (kind, dt)
    m = dz.Model.from_tensors(cfg, t)
    rng = np.random.default_rng(5)
    st = (rng.standard_normal((6, 128, 128)) * 0.1).astype(np.float32)
    conv = (rng.standard_normal((4, cfg.qkv_dim)) * 0.3).astype(np.float32)
    ids = rng.integers(0, cfg.vocab, 96).astype(np.uint32)
    outs = []
    for step in (96, 32):
        ctx = dz.Context(m)
        ctx.set_ssm_state(0, st, conv, 2)
        lg = [ctx.forward_batch(ids[i:i + step], per_pos_logits=True) for i in range(0, 96, step)]
        outs.append((np.concatenate([x.reshape(-1, cfg.vocab) for x in lg]), ctx.get_ssm_state(0)[0]))
    (lc, sc), (lt, s_t) = outs
    assert np.isfinite(lt).all() and np.isfinite(lc).all()
    for i in range(96):
        assert normwise_rel(lc[i], lt[i]) < 2e-5, i
    assert normwise_rel(sc, s_t) < 2e-5
