"""The work a user of nanopd_amd has it do, as cases that can be timed.

One pass is what one attention layer (or one whole engine step) asks of the
public entry points, with new K/V rows stored before they are attended to:

* ``decode``   -- one new token per sequence: ``paged_kv_store`` and
  ``paged_attention_forward`` (the drop-in ops), or over an FP8 pool
  ``paged_kv_store_slots_fp8`` and ``paged_attention_forward_fp8``;
* ``prefill``  -- prompt chunks on a paged prefix: the fused prologue
  ``qk_norm_rope_store`` (or ``paged_kv_store_slots`` for sources that are
  rotated already) and ``paged_prefill_attention`` / ``.._fp8``;
* ``model``    -- ``pack_metadata`` and ``PagedQwen3.forward`` of one mixed
  engine step (a prompt chunk plus the running sequences' decode tokens).

Block tables are slices of a random permutation of the pool (fragmented, as
a serving pool is) and the pool holds a quarter more blocks than are used.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from nanopd_amd import paged_kernels as pk
from nanopd_amd.qwen3 import QWEN2_1_5B, QWEN3_8B, PagedQwen3, StepBatch

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
MODELS = {"qwen3_8b": QWEN3_8B, "qwen2_1.5b": QWEN2_1_5B}
KV_SCALE = 1.0 / 16          # the model's default scale of an FP8 pool
EPS = 1.0e-6
THETA = 1.0e6


def _decode(name, heads, kv_heads, dim, block, dtype, fp8, seqs, ctx_min, ctx_max):
    c = {"op": "decode", "heads": heads, "kv_heads": kv_heads, "dim": dim, "block": block,
         "dtype": dtype, "fp8": fp8, "seqs": seqs, "ctx_min": ctx_min, "ctx_max": ctx_max}
    return dict(c, name=name) if name else c


def _prefill(name, heads, kv_heads, dim, block, dtype, fp8, prologue, seqs, chunk_min, chunk_max,
             prefix_max):
    c = {"op": "prefill", "heads": heads, "kv_heads": kv_heads, "dim": dim, "block": block,
         "dtype": dtype, "fp8": fp8, "prologue": prologue, "seqs": seqs, "chunk_min": chunk_min,
         "chunk_max": chunk_max, "prefix_max": prefix_max}
    return dict(c, name=name) if name else c


def _model(name, model, chunk, prefix, decodes, ctx_min, ctx_max):
    c = {"op": "model", "model": model, "chunk": chunk, "prefix": prefix, "decodes": decodes,
         "ctx_min": ctx_min, "ctx_max": ctx_max}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a few short conversations on a small model: launches and host calls count
        _decode("decode_small", 12, 2, 128, 16, "fp16", False, 4, 17, 511),
        # a full decode batch of the 32-head model
        _decode("decode_batch", 32, 8, 128, 16, "bf16", False, 64, 128, 4096),
        # a handful of long documents
        _decode("decode_long", 32, 8, 128, 16, "bf16", False, 8, 8193, 32769),
        # many short chats at once on a 64-head model
        _decode("decode_many", 64, 8, 128, 16, "bf16", False, 200, 60, 1100),
        # the full decode batch with the pool kept in FP8
        _decode("decode_fp8", 32, 8, 128, 16, "bf16", True, 64, 128, 4096),
        # a head dim off the powers of two
        _decode("decode_d96", 32, 8, 96, 16, "bf16", False, 24, 100, 3000),
        # chunked prefill of four prompts on growing prefixes
        _prefill("prefill_chunks", 32, 8, 128, 16, "bf16", False, "norm", 4, 512, 512, 3072),
        # one long prompt from scratch
        _prefill("prefill_long", 32, 8, 128, 16, "bf16", False, "none", 1, 12000, 12000, 0),
        # short ragged prompts on the small model (q/k without norms)
        _prefill("prefill_short", 12, 2, 128, 16, "fp16", False, "rope", 6, 5, 300, 0),
        # a 64-head model's prompt chunks over an FP8 pool
        _prefill("prefill_fp8", 64, 8, 128, 32, "bf16", True, "norm", 3, 300, 1000, 4096),
        # wide heads
        _prefill("prefill_d256", 16, 8, 256, 16, "bf16", False, "norm", 3, 200, 1024, 1500),
        # a whole engine step: a 512-token chunk and 15 decode tokens
        _model("model_step", "qwen3_8b", 512, 512, 15, 200, 1500),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["decode"] * 5 + ["prefill"] * 5 + ["model"])
    if op == "model":
        chunk = _log(rng, 16, 512)
        return _model(None, rng.choice(["qwen3_8b", "qwen2_1.5b"]), chunk,
                      rng.choice([0, _log(rng, 64, 2048)]), rng.randint(1, 15), 50,
                      _log(rng, 100, 2000))
    heads, kvh = rng.choice([(12, 2), (16, 8), (32, 8), (32, 8), (64, 8), (28, 4)])
    block, dtype = rng.choice([16, 16, 32]), rng.choice(["bf16", "bf16", "fp16"])
    dim = rng.choice([128] * 5 + [64, 96, 256])
    fp8 = rng.random() < 0.25
    if op == "decode":
        if fp8:
            dim = 128            # what FP8 decode takes
        ctx = _log(rng, 64, 32768)
        seqs = _log(rng, 1, max(1, min(256, 200000 // ctx)))
        return _decode(None, heads, kvh, dim, block, dtype, fp8, seqs, max(1, ctx // 16), ctx)
    prologue = rng.choice(["norm", "rope", "none"])
    if dim == 96:                # the fused prologue takes 64, 128 and 256
        prologue = "none"
    chunk = _log(rng, 16, 8192)
    seqs = _log(rng, 1, max(1, min(12, 8192 // chunk)))
    prefix = rng.choice([0, _log(rng, 64, 6000)])
    return _prefill(None, heads, kvh, dim, block, dtype, fp8, prologue, seqs, max(1, chunk // 8),
                    chunk, prefix)


# -- sizes -------------------------------------------------------------------

def _lens(case):
    """Per sequence (new tokens, cached tokens before them), fixed by the case."""
    rng = np.random.default_rng([len(case)] + [v for v in case.values() if type(v) is int])
    if case["op"] == "decode":
        ctx = rng.integers(case["ctx_min"], case["ctx_max"], size=case["seqs"], endpoint=True)
        return [(1, int(n) - 1) for n in ctx]
    if case["op"] == "prefill":
        n = case["seqs"]
        new = rng.integers(case["chunk_min"], case["chunk_max"], size=n, endpoint=True)
        step = case["prefix_max"] // max(1, n - 1) if n > 1 else 0
        pre = [i * step for i in range(n)] if n > 1 else [case["prefix_max"]]
        return [(int(q), int(p)) for q, p in zip(new, pre)]
    ctx = rng.integers(min(case["ctx_min"], case["ctx_max"]), case["ctx_max"],
                       size=case["decodes"], endpoint=True)
    return [(case["chunk"], case["prefix"])] + [(1, int(n)) for n in ctx]


def _shape(case):
    if case["op"] == "model":
        m = MODELS[case["model"]]
        return m.num_heads, m.num_kv_heads, m.head_dim, 16
    return case["heads"], case["kv_heads"], case["dim"], case["block"]


def work(case):
    lens = _lens(case)
    H, KV, D, _ = _shape(case)
    new = sum(q for q, _ in lens)
    old = sum(p for _, p in lens)
    pairs = sum(q * p + q * (q + 1) // 2 for q, p in lens)
    elt = 1 if case.get("fp8") else 2
    kv = 2 * KV * D * elt * (old + new)              # cached rows read, new rows written
    if case["op"] != "model":
        qkv = 2 * (H + 2 * KV) * D * new             # q, k and v of the new tokens
        return {"bytes": kv + qkv + 2 * H * D * new, "flops": 4 * H * D * pairs}
    m = MODELS[case["model"]]
    mats = m.num_layers * ((2 * H + 2 * KV) * D * m.hidden + 3 * m.hidden * m.intermediate)
    head = m.vocab * m.hidden
    rows = len(lens)
    return {"bytes": 2 * (mats + head) + m.num_layers * kv + 4 * rows * m.vocab,
            "flops": 2 * mats * new + 2 * head * rows + m.num_layers * 4 * H * D * pairs}


# -- inputs ------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape, std=1.0, dtype=torch.bfloat16):
    return torch.empty(*shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=g)


def _tables(lens, block, seed):
    """A block table per sequence and the pool's size."""
    need = [(q + p + block - 1) // block for q, p in lens]
    pool = sum(need) + sum(need) // 4 + 1
    perm = np.random.default_rng(seed).permutation(pool)
    out, o = [], 0
    for n in need:
        out.append(perm[o:o + n].astype(np.int32))
        o += n
    return out, pool


def _padded(tables):
    t = np.zeros((len(tables), max(len(x) for x in tables)), dtype=np.int32)
    for i, x in enumerate(tables):
        t[i, :len(x)] = x
    return t


def _dev(a, dtype=np.int32):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=dtype)).to(DEV)


def _fp8(x, scale):
    """e4m3 of x / scale, ties to even."""
    return torch.clamp(x.float() / scale, -448.0, 448.0).to(torch.float8_e4m3fn)


def _inputs(case, seed):
    """The tensors of a decode or prefill case."""
    H, KV, D, bs = _shape(case)
    lens, dt, g = _lens(case), DTYPES[case["dtype"]], _gen(seed)
    tables, pool = _tables(lens, bs, seed)
    T = sum(q for q, _ in lens)
    s = {"lens": lens, "tables": tables, "block_tables": _dev(_padded(tables))}
    pos = np.concatenate([np.arange(p, p + q) for q, p in lens])
    slots = np.concatenate([t[np.arange(p, p + q) // bs] * bs + np.arange(p, p + q) % bs
                            for (q, p), t in zip(lens, tables)])
    s["positions"], s["slots"] = _dev(pos), _dev(slots)
    s["cu"] = _dev(np.concatenate([[0], np.cumsum([q for q, _ in lens])]))
    s["seq_lens"] = _dev([q + p for q, p in lens])
    for k in ("k_cache", "v_cache"):
        c = _randn(g, pool, KV, bs, D, dtype=dt)
        s[k] = _fp8(c, KV_SCALE).view(torch.uint8) if case["fp8"] else c
    if case["fp8"]:
        s["scale"] = torch.full((KV,), KV_SCALE, dtype=torch.float32, device=DEV)
    # rows of the fused projection: q, k and v heads of each token; attention
    # is peaked a little, as trained heads are
    qkv = _randn(g, T, H + 2 * KV, D, dtype=dt)
    if case["op"] == "decode" or case["prologue"] == "none":
        qkv[:, :H] *= 2.0
    s["qkv"] = qkv
    if case["op"] == "prefill" and case["prologue"] == "norm":
        s["q_norm"] = (2.0 + _randn(g, D, std=0.2, dtype=torch.float32)).to(dt)
        s["k_norm"] = (1.0 + _randn(g, D, std=0.2, dtype=torch.float32)).to(dt)
    s["inv_freq"] = 1.0 / (THETA ** (torch.arange(0, D, 2, dtype=torch.float32, device=DEV) / D))
    return s


def _weights(m, g):
    """Random weights of a model, by the names a checkpoint has them under."""
    H, KV, D, E, I = m.num_heads, m.num_kv_heads, m.head_dim, m.hidden, m.intermediate

    def one(n):
        return (1.0 + _randn(g, n, std=0.1, dtype=torch.float32)).to(torch.bfloat16)

    sd = {"model.embed_tokens.weight": _randn(g, m.vocab, E, std=0.02), "model.norm.weight": one(E)}
    if not m.tie_word_embeddings:
        sd["lm_head.weight"] = _randn(g, m.vocab, E, std=0.02)
    for i in range(m.num_layers):
        p = f"model.layers.{i}."
        for nm, rows in (("q", H), ("k", KV), ("v", KV)):
            sd[f"{p}self_attn.{nm}_proj.weight"] = _randn(g, rows * D, E, std=0.02)
            if m.qkv_bias:
                sd[f"{p}self_attn.{nm}_proj.bias"] = _randn(g, rows * D, std=0.02)
        if m.qk_norm:
            sd[p + "self_attn.q_norm.weight"], sd[p + "self_attn.k_norm.weight"] = one(D), one(D)
        sd[p + "self_attn.o_proj.weight"] = _randn(g, E, H * D, std=0.02)
        sd[p + "mlp.gate_proj.weight"] = _randn(g, I, E, std=0.02)
        sd[p + "mlp.up_proj.weight"] = _randn(g, I, E, std=0.02)
        sd[p + "mlp.down_proj.weight"] = _randn(g, E, I, std=0.02)
        sd[p + "input_layernorm.weight"], sd[p + "post_attention_layernorm.weight"] = one(E), one(E)
    return sd


def _model_inputs(case, seed):
    m, g = MODELS[case["model"]], _gen(seed)
    lens = _lens(case)
    tables, pool = _tables(lens, 16, seed)
    sd = _weights(m, g)
    shape = (m.num_layers, pool, m.num_kv_heads, 16, m.head_dim)
    T = sum(q for q, _ in lens)
    return {"lens": lens, "tables": tables, "pool": pool, "sd": sd,
            "k_cache": _randn(g, *shape), "v_cache": _randn(g, *shape),
            "ids": np.random.default_rng(seed + 1).integers(0, m.vocab, size=T)}


def prepare(case, seed):
    if case["op"] == "model":
        i = _model_inputs(case, seed)
        model = PagedQwen3(MODELS[case["model"]], i["pool"], device=DEV)
        model.load_hf_state_dict(i["sd"])
        model.k_cache.copy_(i["k_cache"])
        model.v_cache.copy_(i["v_cache"])
        cu = np.cumsum([q for q, _ in i["lens"]])
        return {"case": case, "model": model, "ids": i["ids"].tolist(),
                "seqs": [(q, p, t.tolist()) for (q, p), t in zip(i["lens"], i["tables"])],
                "rows": [int(x) - 1 for x in cu]}
    s = _inputs(case, seed)
    H, KV, D, bs = _shape(case)
    T = s["qkv"].size(0)
    qkv = s["qkv"]
    s["case"], s["sm_scale"] = case, 1.0 / math.sqrt(D)
    s["out"] = torch.empty(T, H, D, dtype=qkv.dtype, device=DEV)
    s["max_q"] = max(q for q, _ in s["lens"])
    s["max_ctx"] = max(q + p for q, p in s["lens"])
    if case["op"] == "decode" and not case["fp8"]:
        # the drop-in store takes [kv heads, tokens, D] and one table row per token
        s["q"] = qkv[:, :H]
        s["k"] = qkv[:, H:H + KV].transpose(0, 1)
        s["v"] = qkv[:, H + KV:].transpose(0, 1)
    elif case["op"] == "decode" or case["prologue"] == "none":
        s["q"], s["k"], s["v"] = qkv[:, :H], qkv[:, H:H + KV], qkv[:, H + KV:]
    else:
        s["qkv"] = qkv.view(T, -1)
        s["q"] = torch.empty(T, H, D, dtype=qkv.dtype, device=DEV)
    return s


def run(state):
    s = state
    case = s["case"]
    if case["op"] == "model":
        dev = s["model"].device
        meta = pk.pack_metadata(s["seqs"], s["model"].block_size, dev)
        batch = StepBatch(
            input_ids=torch.tensor(s["ids"], dtype=torch.int64).to(dev, non_blocking=True),
            meta=meta, num_prefill_seqs=1, num_prefill_tokens=case["chunk"],
            sample_rows=torch.tensor(s["rows"], dtype=torch.int64).to(dev, non_blocking=True),
            max_prefill_q=case["chunk"])
        logits = s["model"].forward(batch)
        return {"logits": logits, "k_cache": s["model"].k_cache, "v_cache": s["model"].v_cache}
    kc, vc, bt = s["k_cache"], s["v_cache"], s["block_tables"]
    bs, mb = kc.size(2), bt.size(1)
    got = {"out": s["out"], "k_cache": kc, "v_cache": vc}
    if case["op"] == "decode":
        args = (s["out"], s["q"], kc, vc, bt, s["seq_lens"], s["sm_scale"], bs, mb)
        if case["fp8"]:
            pk.paged_kv_store_slots_fp8(kc, vc, s["k"], s["v"], s["slots"], s["scale"], s["scale"])
            pk.paged_attention_forward_fp8(*args, s["scale"], s["scale"])
        else:
            pk.paged_kv_store(kc, vc, s["k"], s["v"], bt, s["positions"])
            pk.paged_attention_forward(*args)
        return got
    scales = (s["scale"], s["scale"]) if case["fp8"] else ()
    if case["prologue"] != "none":
        pk.qk_norm_rope_store(s["q"], kc, vc, s["qkv"], s["slots"], s["positions"], s["inv_freq"],
                              s.get("q_norm"), s.get("k_norm"), EPS, *scales)
        got["q"] = s["q"]
    elif case["fp8"]:
        pk.paged_kv_store_slots_fp8(kc, vc, s["k"], s["v"], s["slots"], *scales)
    else:
        pk.paged_kv_store_slots(kc, vc, s["k"], s["v"], s["slots"])
    args = (s["out"], s["q"], kc, vc, bt, s["cu"], s["seq_lens"], s["sm_scale"], bs, mb, s["max_q"])
    if case["fp8"]:
        pk.paged_prefill_attention_fp8(*args, *scales, s["max_ctx"])
    else:
        pk.paged_prefill_attention(*args, s["max_ctx"])
    return got


# -- what the answers should be ----------------------------------------------

def tolerance(case):
    # about four times the error against exact(): attention rounds its
    # probabilities and its result to the 16-bit type (2e-3 of a bf16 result,
    # 3e-4 of an fp16 one); the prologue rounds q and k before the scores
    # (6e-3, 5e-4); 28 to 36 layers of such steps give logits off by 4e-2 to
    # 5e-2. An FP8 pool's new bytes may round the other way where a 16-bit
    # value sits at a tie.
    if case["op"] == "model":
        return {"rel": 0.15}
    rotated = case["op"] == "decode" or case["prologue"] == "none"
    rel = {("bf16", True): 8e-3, ("bf16", False): 2.5e-2,
           ("fp16", True): 1.2e-3, ("fp16", False): 2.5e-3}[case["dtype"], rotated]
    return {"rel": rel, "differ": 1e-3} if case["fp8"] else {"rel": rel}


def _attend64(q, k, v, first):
    """q [Tq, H, D] at positions first.., k / v [n, KV, D], in 64 bits."""
    Tq, H, D = q.shape
    n, KV = k.shape[:2]
    G = H // KV
    kt = k.permute(1, 2, 0).contiguous()
    vt = v.permute(1, 0, 2).contiguous()
    out = torch.empty(Tq, H, D, dtype=torch.float64, device=q.device)
    rows = max(1, (1 << 28) // (H * n))
    for a in range(0, Tq, rows):
        e = min(Tq, a + rows)
        qq = q[a:e].reshape(e - a, KV, G, D).permute(1, 0, 2, 3).reshape(KV, (e - a) * G, D)
        see = (torch.arange(n, device=q.device)[None, :]
               <= torch.arange(first + a, first + e, device=q.device)[:, None])
        sc = torch.bmm(qq.contiguous(), kt).view(KV, e - a, G, n) / math.sqrt(D)
        sc.masked_fill_(~see[None, :, None, :], -math.inf)
        p = torch.softmax(sc, dim=-1).view(KV, (e - a) * G, n)
        o = torch.bmm(p, vt).view(KV, e - a, G, D)
        out[a:e] = o.permute(1, 0, 2, 3).reshape(e - a, H, D)
    return out


def _rope64(x, positions, inv_freq):
    ang = positions.double()[:, None] * inv_freq.double()[None, :]
    cos, sin = ang.cos()[:, None, :], ang.sin()[:, None, :]
    a, b = x.chunk(2, dim=-1)
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _rms64(x, w):
    y = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w.double()


def _rows(cache, table, n):
    """The first n rows of a sequence, [n, KV, D]."""
    t = torch.from_numpy(table[:(n + cache.size(2) - 1) // cache.size(2)].astype(np.int64)).to(cache.device)
    c = cache[t].permute(0, 2, 1, 3)
    return c.reshape(-1, c.size(2), c.size(3))[:n]


def _put(cache, slots, rows):
    """rows [T, KV, D] at flat slots of cache [blocks, KV, bs, D]."""
    bs, slots = cache.size(2), slots.long()
    cache[slots // bs, :, slots % bs] = rows


def exact(case, seed):
    if case["op"] == "model":
        return _exact_model(case, seed)
    s = _inputs(case, seed)
    H, KV, D, _ = _shape(case)
    dt = DTYPES[case["dtype"]]
    x = s["qkv"].double()
    q, k, v = x[:, :H], x[:, H:H + KV], x[:, H + KV:]
    got = {}
    if case["op"] == "prefill" and case["prologue"] != "none":
        if case["prologue"] == "norm":
            q, k = _rms64(q, s["q_norm"]), _rms64(k, s["k_norm"])
        q, k = (_rope64(t, s["positions"], s["inv_freq"]) for t in (q, k))
        got["q"] = q
    if case["fp8"]:
        # stored bytes, rounded once to the 16-bit type on the way as the ops do
        pools = [s["k_cache"].view(torch.float8_e4m3fn), s["v_cache"].view(torch.float8_e4m3fn)]
        for c, r in zip(pools, (k, v)):
            # (torch has no indexed store of this type: the bytes move as uint8)
            _put(c.view(torch.uint8), s["slots"], _fp8(r.to(dt), KV_SCALE).view(torch.uint8))
        kc, vc = (c.double() * KV_SCALE for c in pools)
        got["k_cache"], got["v_cache"] = (c.view(torch.uint8) for c in pools)
    else:
        kc, vc = s["k_cache"].double(), s["v_cache"].double()
        _put(kc, s["slots"], k)
        _put(vc, s["slots"], v)
        got["k_cache"], got["v_cache"] = kc, vc
    outs, o = [], 0
    for (n, p), t in zip(s["lens"], s["tables"]):
        outs.append(_attend64(q[o:o + n], _rows(kc, t, p + n), _rows(vc, t, p + n), p))
        o += n
    got["out"] = torch.cat(outs)
    return got


def _exact_model(case, seed):
    m, i = MODELS[case["model"]], _model_inputs(case, seed)
    H, KV, D, E = m.num_heads, m.num_kv_heads, m.head_dim, m.hidden
    sd, lens, tables = i["sd"], i["lens"], i["tables"]
    pos = _dev(np.concatenate([np.arange(p, p + q) for q, p in lens]))
    slots = _dev(np.concatenate([t[np.arange(p, p + q) // 16] * 16 + np.arange(p, p + q) % 16
                                 for (q, p), t in zip(lens, tables)]))
    inv = 1.0 / (m.rope_theta ** (torch.arange(0, D, 2, dtype=torch.float64, device=DEV) / D))
    kc, vc = i["k_cache"].double(), i["v_cache"].double()
    x = sd["model.embed_tokens.weight"][torch.from_numpy(i["ids"]).to(DEV)].double()
    T = x.size(0)
    for li in range(m.num_layers):
        def w(name):
            return sd[f"model.layers.{li}.{name}"].double()

        h = _rms64(x, w("input_layernorm.weight"))
        q, k, v = (h @ w(f"self_attn.{n}_proj.weight").t() for n in "qkv")
        if m.qkv_bias:
            q, k, v = (y + w(f"self_attn.{n}_proj.bias") for n, y in zip("qkv", (q, k, v)))
        q, k, v = q.view(T, H, D), k.view(T, KV, D), v.view(T, KV, D)
        if m.qk_norm:
            q, k = _rms64(q, w("self_attn.q_norm.weight")), _rms64(k, w("self_attn.k_norm.weight"))
        q, k = _rope64(q, pos, inv), _rope64(k, pos, inv)
        _put(kc[li], slots, k)
        _put(vc[li], slots, v)
        outs, o = [], 0
        for (n, p), t in zip(lens, tables):
            outs.append(_attend64(q[o:o + n], _rows(kc[li], t, p + n), _rows(vc[li], t, p + n), p))
            o += n
        x = x + torch.cat(outs).view(T, H * D) @ w("self_attn.o_proj.weight").t()
        h = _rms64(x, w("post_attention_layernorm.weight"))
        gate, up = h @ w("mlp.gate_proj.weight").t(), h @ w("mlp.up_proj.weight").t()
        x = x + (gate * torch.sigmoid(gate) * up) @ w("mlp.down_proj.weight").t()
    rows = torch.from_numpy(np.cumsum([q for q, _ in lens]) - 1).to(DEV)
    xs = _rms64(x[rows], sd["model.norm.weight"])
    head = sd["model.embed_tokens.weight" if m.tie_word_embeddings else "lm_head.weight"]
    return {"logits": xs @ head.double().t(), "k_cache": kc, "v_cache": vc}
