"""Workloads of the Q1_0 token loop, each through the public entry points of daiza_amd.

Shapes are those of the 27B configuration (Config.bonsai27b) and of the tests: single Q1_0 products,
one DeltaNet or attention layer-step, a four-layer block (three DeltaNet layers and one attention
layer, each with its MLP, then the head) in prefill and in speculative verify, and the whole
64-layer model in decode.

A case is a dict of plain values; `op` names the entry point:
  matvec     dz_q1_0_matvec_dev on device vectors, `mats` matrices one after another
  batch      Q1_0Matrix.matvec_batch_into_slice on host arrays, n columns
  layer      dz_ctx_mixer_step_dev, `steps` tokens through one layer over a context
  prefill    Context.forward_batch of n tokens through the block after `start` cached positions
  verify     Context.verify_forward of k drafts through the block, then verify_commit of half of them
  decode     Context.decode_greedy / decode_sample of n tokens through the 64-layer model
"""
import ctypes
import math

import numpy as np
import torch

import daiza_amd as dz

WEIGHT_SEED = 0xDA1A0004  # the whole model's weights; prompts, states and drafts come from the case's seed
VOCAB_BLOCK = 2048


def listed():
    return [
        # the smallest product a token makes (alpha and beta rows of a reduced stack): launch latency
        dict(name="matvec_small", op="matvec", rows=1024, cols=512, mats=1),
        # the FFN up-projection of eight layers in turn, as a token passes them: weights come from HBM
        dict(name="matvec_ffn", op="matvec", rows=17408, cols=5120, mats=8),
        # the head's product over the whole vocabulary
        dict(name="matvec_head", op="matvec", rows=248320, cols=5120, mats=1),
        # matvec_batch as a caller with host arrays makes it: the eight drafts of a verify step
        dict(name="batch_8", op="batch", rows=17408, cols=5120, n=8),
        # one DeltaNet layer over 16 tokens
        dict(name="deltanet_layer", op="layer", attn=False, ctx=0, steps=16),
        # one attention layer over 16 tokens, at an ordinary and at a long context
        dict(name="attention_layer_4096", op="layer", attn=True, ctx=4096, steps=16),
        dict(name="attention_layer_32768", op="layer", attn=True, ctx=32768, steps=16),
        # a long prompt into an empty context
        dict(name="prefill_1024", op="prefill", start=0, n=1024),
        # the next turn of a conversation: a ragged number of tokens behind a long cached prefix
        dict(name="prefill_333_at_7000", op="prefill", start=7000, n=333),
        # one speculative step: eight drafts over a long context
        dict(name="verify_8_at_8192", op="verify", ctx=8192, k=8),
        # the token loop of the whole model, greedy and sampled
        dict(name="decode_greedy_27b", op="decode", prompt=1024, n=16, sample=False),
        dict(name="decode_sample_27b", op="decode", prompt=256, n=16, sample=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["matvec", "matvec", "batch", "layer", "layer", "prefill", "prefill", "verify", "decode"])
    if op == "matvec":
        rows, cols = _log_int(rng, 64, 248320), 128 * _log_int(rng, 1, 136)
        rows = min(rows, 248320 * 5120 // cols)
        return dict(op=op, rows=rows, cols=cols, mats=rng.randint(1, max(1, min(8, 8 * 17408 * 5120 // (rows * cols)))))
    if op == "batch":
        return dict(op=op, rows=_log_int(rng, 64, 17408), cols=128 * _log_int(rng, 1, 136), n=_log_int(rng, 1, 256))
    if op == "layer":
        attn = rng.random() < 0.7
        return dict(op=op, attn=attn, ctx=_log_int(rng, 64, 32768) if attn else 0, steps=rng.randint(2, 16))
    if op == "prefill":
        return dict(op=op, start=0 if rng.random() < 0.5 else _log_int(rng, 64, 12000), n=_log_int(rng, 1, 1024))
    if op == "verify":
        return dict(op=op, ctx=_log_int(rng, 64, 12000), k=rng.randint(1, 16))
    return dict(op=op, prompt=_log_int(rng, 32, 1024), n=rng.randint(2, 16), sample=rng.random() < 0.5)


# ---------------------------------------------------------------- inputs


def _gen(seed, *tag):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + sum((i + 1) * 7919 * int(t) for i, t in enumerate(tag))) & 0x7FFFFFFFFFFF)
    return g


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * std


def _q1(g, rows, cols):
    """Q1_0 bytes [rows][cols/128][18] (uint8, device): random sign bits, scale f16(|N(0,1)| * 0.02)."""
    out = torch.empty(rows, cols // 128, 18, dtype=torch.uint8, device="cuda")
    out[:, :, 2:] = torch.randint(0, 256, (rows, cols // 128, 16), generator=g, device="cuda", dtype=torch.uint8)
    sc = (_normal(g, rows, cols // 128).abs() * 0.02).to(torch.float16)
    out[:, :, :2] = sc.view(torch.uint8).view(rows, cols // 128, 2)
    return out


def _q1_product(q, x):
    """x[n][cols] (float64) times the transposed matrix of Q1_0 bytes q, in 64 bits."""
    rows, groups = q.shape[0], q.shape[1]
    out = torch.empty(x.shape[0], rows, dtype=torch.float64, device="cuda")
    step = max(1, (1 << 26) // (groups * 128))
    bit = torch.arange(8, device="cuda", dtype=torch.uint8)
    for r in range(0, rows, step):
        b = q[r:r + step]
        sc = b[:, :, :2].contiguous().view(torch.float16).to(torch.float64)
        w = ((b[:, :, 2:, None] >> bit) & 1).to(torch.float64).mul_(2.0).sub_(1.0).flatten(2) * sc
        out[:, r:r + step] = x @ w.flatten(1).t()
    return out


def _block_config(max_ctx, n_layers=4, interval=4, vocab=VOCAB_BLOCK):
    c = dz.Config.bonsai27b(max_ctx=max_ctx)
    c.n_layers, c.full_attn_interval, c.vocab = n_layers, interval, vocab
    return c


def _is_attn(c, i):
    return i % c.full_attn_interval == c.full_attn_interval - 1


def _block_weights(c, seed):
    """{GGUF name: device tensor}: Q1_0 bytes [rows][groups][18], float32 vectors, an f16 embedding."""
    w = {}
    H, F, hd = c.hidden, c.ffn, c.ssm_state
    kd, inner = c.ssm_k_heads * hd, c.ssm_v_heads * hd
    qd, kvd = c.n_head * c.head_dim, c.n_head_kv * c.head_dim

    def norm(g, n):
        return torch.rand(n, generator=g, device="cuda") * 0.4 + 0.8

    for i in range(c.n_layers):
        g, b = _gen(seed, 1, i), "blk.%d." % i
        w[b + "attn_norm.weight"], w[b + "post_attention_norm.weight"] = norm(g, H), norm(g, H)
        w[b + "ffn_gate.weight"], w[b + "ffn_up.weight"] = _q1(g, F, H), _q1(g, F, H)
        w[b + "ffn_down.weight"] = _q1(g, H, F)
        if _is_attn(c, i):
            w[b + "attn_q.weight"] = _q1(g, 2 * qd, H)
            w[b + "attn_k.weight"], w[b + "attn_v.weight"] = _q1(g, kvd, H), _q1(g, kvd, H)
            w[b + "attn_output.weight"] = _q1(g, H, qd)
            w[b + "attn_q_norm.weight"], w[b + "attn_k_norm.weight"] = norm(g, c.head_dim), norm(g, c.head_dim)
        else:
            w[b + "attn_qkv.weight"], w[b + "attn_gate.weight"] = _q1(g, 2 * kd + inner, H), _q1(g, inner, H)
            w[b + "ssm_alpha.weight"], w[b + "ssm_beta.weight"] = _q1(g, c.ssm_v_heads, H), _q1(g, c.ssm_v_heads, H)
            w[b + "ssm_out.weight"] = _q1(g, H, inner)
            w[b + "ssm_conv1d.weight"] = _normal(g, 2 * kd + inner, c.ssm_conv_kernel, std=0.25)
            w[b + "ssm_a"] = -torch.exp(torch.rand(c.ssm_v_heads, generator=g, device="cuda") * 2 - 1)
            w[b + "ssm_dt.bias"] = _normal(g, c.ssm_v_heads, std=0.1)
            w[b + "ssm_norm.weight"] = norm(g, hd)
    g = _gen(seed, 2)
    w["output_norm.weight"], w["output.weight"] = norm(g, H), _q1(g, c.vocab, H)
    # values of the f16 grid in [-1, 1] away from its subnormals
    w["token_embd.weight"] = (torch.randint(-1024, 1025, (c.vocab, H), generator=g, device="cuda") / 1024).to(torch.float16)
    return w


def _block_model(c, w):
    kinds = {torch.uint8: dz.GGUF_Q1_0, torch.float32: dz.GGUF_F32, torch.float16: dz.GGUF_F16}
    return dz.Model.from_tensors(c, {k: (kinds[t.dtype], t.cpu().numpy()) for k, t in w.items()})


def _block_state(c, seed, length):
    """{layer: (K, V) [kv heads][length][dim]} or {layer: (S [v heads][128][128], conv rows [4][channels])}."""
    st = {}
    for i in range(c.n_layers):
        g = _gen(seed, 3, i)
        if _is_attn(c, i):
            # keys of twice the unit length: scores of a spread that lets some positions stand out
            st[i] = (_normal(g, c.n_head_kv, length, c.head_dim, std=2.0), _normal(g, c.n_head_kv, length, c.head_dim))
        else:
            st[i] = (_normal(g, c.ssm_v_heads, c.ssm_state, c.ssm_state, std=0.02), _normal(g, 4, c.qkv_dim, std=0.1))
    return st


def _load_state(ctx, c, st, length):
    for i, (a, b) in st.items():
        if _is_attn(c, i):
            if length:
                ctx.set_kv(i, a.cpu().numpy(), b.cpu().numpy())
        else:
            ctx.set_ssm_state(i, a.cpu().numpy(), b.cpu().numpy(), 0)
    ctx.set_pos(length)


def _tokens(seed, n, vocab):
    return np.random.default_rng([int(seed), 17]).integers(0, vocab, n).astype(np.uint32)


_whole = {}


def _whole_model():
    """The 64-layer model, its weights resident once per program."""
    if not _whole:
        cfg = dz.Config.bonsai27b(max_ctx=1088)
        _whole["cfg"], _whole["model"] = cfg, dz.Model.synthetic(cfg, WEIGHT_SEED)
    return _whole["cfg"], _whole["model"]


def _layer_config(case):
    return _block_config(max(64, case["ctx"]) + case["steps"], n_layers=1, interval=1 if case["attn"] else 4, vocab=1024)


def _layer_input(case, c, seed):
    """Hidden vectors of the size of what a layer adds to them (the layer normalises them first)."""
    return _normal(_gen(seed, 6), case["steps"], c.hidden, std=0.1)


def prepare(case, seed):
    if dz.lib().dz_device_init(0) != 0:
        raise RuntimeError(dz.lib().dz_last_error().decode())
    op = case["op"]
    if op == "matvec":
        g = _gen(seed, 5)
        mats = [dz.Q1_0Matrix(_q1(g, case["rows"], case["cols"]).cpu().numpy().reshape(-1), case["rows"], case["cols"])
                for _ in range(case["mats"])]
        x = _normal(g, case["mats"], case["cols"])
        return dict(case, m=mats, x=x, y=torch.empty(case["mats"], case["rows"], device="cuda"))
    if op == "batch":
        g = _gen(seed, 5)
        m = dz.Q1_0Matrix(_q1(g, case["rows"], case["cols"]).cpu().numpy().reshape(-1), case["rows"], case["cols"])
        x = _normal(g, case["n"], case["cols"]).cpu().numpy()
        return dict(case, m=m, x=x, y=np.empty((case["n"], case["rows"]), np.float32))
    if op == "layer":
        c = _layer_config(case)
        model = _block_model(c, _block_weights(c, seed))
        ctx = dz.Context(model)
        _load_state(ctx, c, _block_state(c, seed, case["ctx"]), case["ctx"])
        h = _layer_input(case, c, seed)
        return dict(case, ctx=ctx, model=model, start=case["ctx"], h=h, out=torch.empty_like(h))
    if op == "prefill":
        c = _block_config(case["start"] + case["n"])
        model = _block_model(c, _block_weights(c, seed))
        ctx, base = dz.Context(model), dz.Context(model) if case["start"] else None
        if base is not None:
            _load_state(base, c, _block_state(c, seed, case["start"]), case["start"])
        return dict(case, ctx=ctx, base=base, model=model, ids=_tokens(seed, case["n"], c.vocab))
    if op == "verify":
        c = _block_config(case["ctx"] + case["k"])
        model = _block_model(c, _block_weights(c, seed))
        ctx = dz.Context(model)
        _load_state(ctx, c, _block_state(c, seed, case["ctx"]), case["ctx"])
        return dict(case, ctx=ctx, model=model, start=case["ctx"], draft=_tokens(seed, case["k"], c.vocab))
    c, model = _whole_model()
    base, ctx = dz.Context(model), dz.Context(model)
    ids = _tokens(seed, case["prompt"], c.vocab)
    first = int(np.argmax(base.forward_batch(ids)))
    return dict(case, ctx=ctx, base=base, first=first, seed=int(seed) & 0xFFFFFFFF)


def run(s):
    op = s["op"]
    if op == "matvec":
        x, y, L = s["x"], s["y"], dz.lib()
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        for i, m in enumerate(s["m"]):
            rc = L.dz_q1_0_matvec_dev(m._h, x.data_ptr() + i * x.stride(0) * 4, y.data_ptr() + i * y.stride(0) * 4, 0, stream)
            if rc != 0:
                raise dz.DaizaError(rc, L.dz_last_error().decode())
        return y
    if op == "batch":
        s["m"].matvec_batch_into_slice(s["x"], s["n"], s["y"])
        return s["y"]
    ctx = s["ctx"]
    if op == "layer":
        L, h, out = dz.lib(), s["h"], s["out"]
        if ctx.pos != s["start"]:
            ctx.set_pos(s["start"])
        for t in range(s["steps"]):
            rc = L.dz_ctx_mixer_step_dev(ctx._h, 0, h.data_ptr() + t * h.stride(0) * 4, out.data_ptr() + t * out.stride(0) * 4)
            if rc != 0:
                raise dz.DaizaError(rc, L.dz_last_error().decode())
        return out
    if op == "prefill":
        if s["base"] is None:
            ctx.reset()
        else:
            ctx.copy_state_from(s["base"])
        return ctx.forward_batch(s["ids"])
    if op == "verify":
        if ctx.pos != s["start"]:
            ctx.kv_truncate(s["start"])
        logits = ctx.verify_forward(s["draft"])
        ctx.verify_commit(s["k"] // 2)
        return logits
    ctx.copy_state_from(s["base"])
    if s["sample"]:
        toks = ctx.decode_sample(s["first"], s["n"], dz.SamplingParams(0.7, 20, 0.95), dz.LcgRng(s["seed"]))
    else:
        toks = ctx.decode_greedy(s["first"], s["n"])
    return {"tokens": toks.astype(np.int64), "logits": ctx.logits()}


# ---------------------------------------------------------------- the work of a pass


def _q1_bytes(rows, cols):
    return rows * (cols // 128) * 18


def _layer_shapes(c, i):
    """(rows, cols) of the mixer's products of layer i."""
    hd = c.ssm_state
    inner, qd, kvd = c.ssm_v_heads * hd, c.n_head * c.head_dim, c.n_head_kv * c.head_dim
    if _is_attn(c, i):
        return [(2 * qd + 2 * kvd, c.hidden), (c.hidden, qd)]
    return [(c.qkv_dim + inner + 2 * c.ssm_v_heads, c.hidden), (c.hidden, inner)]


def _forward_work(c, start, n, heads, mlp=True, per_token=False):
    """Bytes and operations of n tokens after `start` cached positions: weights read once (once per token
    in a token loop), states read and written, cached rows read and new ones written."""
    passes, byts, flops = n if per_token else 1, 0, 0
    kv_row, state = 2 * c.n_head_kv * c.head_dim * 4, c.ssm_v_heads * c.ssm_state ** 2
    seen = sum(start + t + 1 for t in range(n))
    for i in range(c.n_layers):
        shapes = _layer_shapes(c, i) + ([(2 * c.ffn, c.hidden), (c.hidden, c.ffn)] if mlp else [])
        byts += passes * sum(_q1_bytes(r, k) for r, k in shapes)
        flops += 2 * n * sum(r * k for r, k in shapes)
        if _is_attn(c, i):
            byts += kv_row * (n + (seen if per_token else start))
            flops += 4 * c.n_head * c.head_dim * seen
        else:
            byts += passes * (2 * state * 4 + 8 * c.qkv_dim * 4)
            flops += n * 7 * state
    if heads:
        byts += (passes if per_token else 1) * _q1_bytes(c.vocab, c.hidden) + heads * c.vocab * 4 + n * c.hidden * 2
        flops += 2 * heads * c.vocab * c.hidden
    else:
        byts += n * 2 * c.hidden * 4
    return {"bytes": byts, "flops": flops}


def work(case):
    op = case["op"]
    if op in ("matvec", "batch"):
        n, mats = case.get("n", 1), case.get("mats", 1)
        return {"bytes": mats * (_q1_bytes(case["rows"], case["cols"]) + 4 * n * (case["rows"] + case["cols"])),
                "flops": 2 * mats * n * case["rows"] * case["cols"]}
    if op == "layer":
        return _forward_work(_layer_config(case), case["ctx"], case["steps"], 0, mlp=False, per_token=True)
    if op == "prefill":
        return _forward_work(_block_config(case["start"] + case["n"]), case["start"], case["n"], 1)
    if op == "verify":
        return _forward_work(_block_config(case["ctx"] + case["k"]), case["ctx"], case["k"], case["k"])
    return _forward_work(dz.Config.bonsai27b(max_ctx=1088), case["prompt"], case["n"], case["n"], per_token=True)


def tolerance(case):
    # 32-bit sums in another order: about four times what each shows against 64 bits (the whole model:
    # against its kernel-per-phase form)
    return {"matvec": {"rel": 1e-6, "max": 1e-5}, "batch": {"rel": 1e-6, "max": 1e-5},
            "layer": {"rel": 2e-6, "max": 2e-5}, "prefill": {"rel": 2e-5, "max": 1e-4},
            "verify": {"rel": 8e-6, "max": 4e-5}, "decode": {"rel": 2.5e-5, "max": 1.5e-4}}[case["op"]]


# ---------------------------------------------------------------- the same in 64 bits


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _rope(x, c, pos):
    """The partial rotation of x[n][heads][dim] at positions pos[n]: pairs (d, d + half), both terms added;
    the angle is the 32-bit product of position and frequency."""
    half = c.rope_dim // 2
    e = np.arange(half, dtype=np.float32) * np.float32(2) / np.float32(c.rope_dim)
    freq = np.float32(1) / np.power(np.float64(c.rope_base), e.astype(np.float64)).astype(np.float32)
    th = torch.from_numpy((pos.astype(np.float32)[:, None] * freq).astype(np.float64)).cuda()[:, None]
    x1, x2 = x[..., :half], x[..., half:2 * half]
    co, si = torch.cos(th), torch.sin(th)
    return torch.cat([x1 * co + x2 * si, x2 * co + x1 * si, x[..., 2 * half:]], -1)


def _deltanet(c, w, b, st, h):
    hd, nk, nv = c.ssm_state, c.ssm_k_heads, c.ssm_v_heads
    n, kd = h.shape[0], nk * hd
    x = _rms(h, w[b + "attn_norm.weight"], c.rms_eps)
    qkv = _q1_product(w[b + "attn_qkv.weight"], x)
    z = _q1_product(w[b + "attn_gate.weight"], x)
    al, be = _q1_product(w[b + "ssm_alpha.weight"], x), _q1_product(w[b + "ssm_beta.weight"], x)
    hist = torch.cat([st[1].double()[1:], qkv])  # three rows before the first token
    cw = w[b + "ssm_conv1d.weight"].double()
    conv = torch.nn.functional.silu(sum(hist[t:t + n] * cw[:, t] for t in range(4)))
    q, k, v = conv[:, :kd].view(n, nk, hd), conv[:, kd:2 * kd].view(n, nk, hd), conv[:, 2 * kd:].view(n, nv, hd)
    q = q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) / math.sqrt(hd)
    k = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    rep = torch.arange(nv, device="cuda") % nk
    q, k = q[:, rep], k[:, rep]
    decay = torch.exp(w[b + "ssm_a"].double() * torch.nn.functional.softplus(al + w[b + "ssm_dt.bias"].double()))
    beta, S, y = torch.sigmoid(be), st[0].double(), torch.empty_like(v)
    for t in range(n):
        S = S * decay[t, :, None, None]
        d = (v[t] - (S @ k[t, :, :, None])[..., 0]) * beta[t, :, None]
        S = S + d[:, :, None] * k[t, :, None, :]
        y[t] = (S @ q[t, :, :, None])[..., 0]
    y = _rms(y, w[b + "ssm_norm.weight"], c.rms_eps) * torch.nn.functional.silu(z).view(n, nv, hd)
    return h + _q1_product(w[b + "ssm_out.weight"], y.flatten(1))


def _attention(c, w, b, st, h, start):
    hd, nq, nkv = c.head_dim, c.n_head, c.n_head_kv
    n, grp = h.shape[0], c.n_head // c.n_head_kv
    pos = np.arange(start, start + n)
    x = _rms(h, w[b + "attn_norm.weight"], c.rms_eps)
    qg = _q1_product(w[b + "attn_q.weight"], x).view(n, nq, 2, hd)
    k = _q1_product(w[b + "attn_k.weight"], x).view(n, nkv, hd)
    v = _q1_product(w[b + "attn_v.weight"], x).view(n, nkv, hd)
    q = _rope(_rms(qg[:, :, 0], w[b + "attn_q_norm.weight"], c.rms_eps), c, pos) / math.sqrt(hd)
    k = _rope(_rms(k, w[b + "attn_k_norm.weight"], c.rms_eps), c, pos)
    o = torch.empty(n, nq, hd, dtype=torch.float64, device="cuda")
    ahead = torch.arange(start + n, device="cuda")[None] > torch.from_numpy(pos).cuda()[:, None]
    for g in range(nkv):
        kk, vv = torch.cat([st[0][g].double(), k[:, g]]), torch.cat([st[1][g].double(), v[:, g]])
        for qh in range(g * grp, (g + 1) * grp):
            o[:, qh] = torch.softmax((q[:, qh] @ kk.t()).masked_fill(ahead, -math.inf), -1) @ vv
    o = o * torch.sigmoid(qg[:, :, 1])
    return h + _q1_product(w[b + "attn_output.weight"], o.flatten(1))


def _mixer(c, w, st, i, h, start):
    b = "blk.%d." % i
    return _attention(c, w, b, st[i], h, start) if _is_attn(c, i) else _deltanet(c, w, b, st[i], h)


def _block(c, w, st, ids, start, heads):
    h = w["token_embd.weight"][torch.from_numpy(ids.astype(np.int64)).cuda()].double()
    for i in range(c.n_layers):
        b = "blk.%d." % i
        h = _mixer(c, w, st, i, h, start)
        x = _rms(h, w[b + "post_attention_norm.weight"], c.rms_eps)
        u = torch.nn.functional.silu(_q1_product(w[b + "ffn_gate.weight"], x)) * _q1_product(w[b + "ffn_up.weight"], x)
        h = h + _q1_product(w[b + "ffn_down.weight"], u)
    return _q1_product(w["output.weight"], _rms(h[-heads:], w["output_norm.weight"], c.rms_eps))


def _zero_state(c):
    return {i: tuple(torch.zeros_like(t) for t in p) for i, p in _block_state(c, 0, 0).items()}


def exact(case, seed):
    op = case["op"]
    if op in ("matvec", "batch"):
        g = _gen(seed, 5)
        n = case.get("n", 1)
        q = [_q1(g, case["rows"], case["cols"]) for _ in range(case.get("mats", 1))]
        if op == "batch":
            return _q1_product(q[0], _normal(g, n, case["cols"]).double()).cpu().numpy()
        x = _normal(g, case["mats"], case["cols"]).double()
        return torch.cat([_q1_product(m, x[i:i + 1]) for i, m in enumerate(q)])
    if op == "layer":
        c = _layer_config(case)
        h = _layer_input(case, c, seed).double()
        return _mixer(c, _block_weights(c, seed), _block_state(c, seed, case["ctx"]), 0, h, case["ctx"])
    if op == "prefill":
        c = _block_config(case["start"] + case["n"])
        st = _block_state(c, seed, case["start"]) if case["start"] else _zero_state(c)
        return _block(c, _block_weights(c, seed), st, _tokens(seed, case["n"], c.vocab), case["start"], 1)[0].cpu().numpy()
    if op == "verify":
        c = _block_config(case["ctx"] + case["k"])
        return _block(c, _block_weights(c, seed), _block_state(c, seed, case["ctx"]), _tokens(seed, case["k"], c.vocab),
                      case["ctx"], case["k"]).cpu().numpy()
    return None  # the whole model takes longer than the blocks that it is made of
