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
    cfg = dz.Config.small(n_layers=1, vocab=128, embd_f16=1, **kw)
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
