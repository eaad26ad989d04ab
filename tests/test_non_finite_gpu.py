"""Causality for infinities and NaN: a token whose embedding holds one makes its own results and those of the
tokens behind it NaN, and leaves every token before it as it is, bit for bit, in the n-token forward and in
verify.  (The matrix instructions multiply what a token does not see by 0, which is NaN for such values.)"""
import numpy as np
import pytest

from named_tensors import named_tensors

pytestmark = pytest.mark.gpu

SEED = 0xDA1A0024
BAD = 7


def _model(dz, oracle, value, **kw):
    cfg = dz.Config.small(**{"n_layers": 1, "vocab": 128, "embd_f16": 1, **kw})
    t = named_tensors(oracle, oracle.Model(cfg, SEED), cfg, SEED)
    kind, emb = t["token_embd.weight"]
    emb = emb.reshape(cfg.vocab, cfg.hidden).copy()
    emb[BAD, 77] = np.float16(value).view(np.uint16)
    t["token_embd.weight"] = (kind, emb)
    return cfg, dz.Model.from_tensors(cfg, t)


def _check(run, n, at, rng):
    ids = rng.integers(BAD + 1, 128, n).astype(np.uint32)
    want = run(ids)
    assert np.isfinite(want).all()
    ids[at] = BAD
    got = run(ids)
    assert np.array_equal(got[:at], want[:at])
    assert np.isnan(got[at:]).all()


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("nq,nkv,start,n,at", [
    (2, 2, 0, 40, 25),        # group 1: a row tile and a chunk per block
    (6, 1, 300, 70, 3),       # group 6: several tiles and chunks
    (6, 1, 0, 33, 32),        # the last token
    (3, 1, 0, 128, 17),       # tokens behind a block of 16 positions
    (8, 1, 16500, 100, 49),   # long chunks (the next block's scores formed ahead), merged
])
def test_attention(dz, oracle, value, nq, nkv, start, n, at):
    cfg, m = _model(dz, oracle, value, n_head=nq, n_head_kv=nkv, full_attn_interval=1, max_ctx=start + n)
    rng = np.random.default_rng(n)
    k, v = (rng.standard_normal((nkv, max(1, start), cfg.head_dim), dtype=np.float32) for _ in range(2))

    def forward(ids):
        ctx = dz.Context(m)
        if start:
            ctx.set_kv(0, k, v)
            ctx.set_pos(start)
        return ctx.forward_batch(ids, per_pos_logits=True)

    _check(forward, n, at, rng)
    if n > 16:
        n, at = 16, at % 16

    def verify(ids):
        ctx = dz.Context(m)
        if start:
            ctx.set_kv(0, k, v)
            ctx.set_pos(start)
        return ctx.verify_forward(ids)

    _check(verify, n, at, rng)


@pytest.mark.parametrize("n,at", [
    (40, 25), (40, 16), (40, 31), (40, 32),  # the first chunk's second tile, its ends, and the chunk behind it
    (128, 48), (128, 3), (33, 32),           # a tile's first token; an early one; a lone last token
    (32, 20), (16, 9), (5, 2),               # the token-by-token kernel
])
def test_delta_rule(dz, oracle, n, at):
    cfg, m = _model(dz, oracle, np.inf, ssm_k_heads=2, ssm_v_heads=6, max_ctx=160)
    rng = np.random.default_rng(n + at)
    st = (rng.standard_normal((6, 128, 128)) * 0.1).astype(np.float32)
    conv = (rng.standard_normal((4, cfg.qkv_dim)) * 0.3).astype(np.float32)

    def run(call):
        def f(ids):
            ctx = dz.Context(m)
            ctx.set_ssm_state(0, st, conv, 2)
            return call(ctx, ids)
        return f

    _check(run(lambda ctx, ids: ctx.forward_batch(ids, per_pos_logits=True)), n, at, rng)
    _check(run(lambda ctx, ids: ctx.verify_forward(ids)), n, at, rng)


def test_value_of_one_head(dz, oracle):
    """A value that overflows in one v-head (a huge conv weight behind a large token) while keys, queries and gates
    stay finite: the tokens before it are untouched, and so is every other v-head's state."""
    cfg = dz.Config.small(n_layers=1, vocab=128, ssm_k_heads=1, ssm_v_heads=2, max_ctx=64)
    t = named_tensors(oracle, oracle.Model(cfg, SEED), cfg, SEED)
    kind, w = t["blk.0.ssm_conv1d.weight"]
    w = w.copy()
    w[2 * 128 + 5] = [0, 0, 0, 3e38]  # value 5 of v-head 0, the current token's tap
    t["blk.0.ssm_conv1d.weight"] = (kind, w)
    m = dz.Model.from_tensors(cfg, t)
    rng = np.random.default_rng(4)
    ids = rng.integers(0, 128, 64).astype(np.uint32)
    out = {}
    for step in (64, 32):  # chunks, and the token-by-token kernel
        ctx = dz.Context(m)
        lg = [ctx.forward_batch(ids[i:i + step], per_pos_logits=True) for i in range(0, 64, step)]
        out[step] = (np.concatenate(lg), ctx.get_ssm_state(0)[0])
    (lc, sc), (lt, s_t) = out[64], out[32]
    assert np.isnan(lt).any()
    assert np.array_equal(np.isfinite(lc).all(1), np.isfinite(lt).all(1))
    assert np.array_equal(np.isfinite(sc), np.isfinite(s_t))
    ok = np.isfinite(s_t)
    assert not ok[0, 5].any() and ok[1].all()
    assert np.abs(sc[ok] - s_t[ok]).max() < 2e-5 * np.abs(s_t[ok]).max()


def test_hybrid_stack(dz, oracle):
    cfg, m = _model(dz, oracle, -np.inf, n_layers=4, max_ctx=160)
    rng = np.random.default_rng(2)
    _check(lambda ids: dz.Context(m).forward_batch(ids, per_pos_logits=True), 128, 77, rng)
    _check(lambda ids: dz.Context(m).verify_forward(ids), 8, 3, rng)
