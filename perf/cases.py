"""The framework's work, as timed cases: what is called, on which inputs, and how exact it must be.

A case is a dict of plain values; `kind` names the entry point that it goes through:

  assemble  _hip.rope_assemble: re-rotate and gather cached blocks into one request's KV cache
  select    _hip.dev_score + _hip.topk_select: the rows of a context that are worth recomputing
  attn      _hip.subset_attn: attention of a row set over a KV cache (causal prefill, packed cold
            documents, recomputed rows)
  layer     blend._layer_subset: one decoder layer recomputed for a row set of a cached context
  append    Engine.decode: one generated token, or a follow-up turn of several, on a request's cache
  request   Engine.prefill: a whole request, its documents cached (warm) or not (cold)

Model shapes are the presets of tread_amd.model with random weights; `layers` cuts the depth where
one call of the full model says nothing that a few layers do not.
"""
import math
import random

import torch

from tread_amd import BlockStore, Engine, _hip, blend
from tread_amd.model import preset, synthetic_model

SYSTEM = 64  # tokens of the system prompt that every request shape of this repository starts with


# ------------------------------------------------------------------------------------------ cases

def listed():
    return [
        # The smallest call on the path: four short documents of a small model gathered into a
        # request's cache. A launch and its preparation, little else.
        dict(name="assemble_small", kind="assemble", model="qwen2.5-0.5b", docs=4, doc_len=256, ragged=False),
        # The largest gather: 32 documents of a 7B-shaped model, 3.7 GB through HBM.
        dict(name="assemble_32k", kind="assemble", model="qwen2.5-7b", docs=32, doc_len=1000, ragged=False),
        # Choosing the rows to recompute out of a 32k context (the score and the selection that
        # every request with recompute waits for).
        dict(name="select_32k", kind="select", model="qwen2.5-7b", rows=32000, ratio=0.2),
        # Attention of a full prefill at head_dim 64 (the uncached request of the small model).
        dict(name="attn_causal_8k", kind="attn", model="qwen2.5-0.5b", form="causal", rows=8096, keys=8096),
        # Attention of documents that were not cached: packed in one prefill, each seeing the
        # shared prefix and itself, ragged lengths, at the 70B shape.
        dict(name="attn_cold_docs", kind="attn", model="llama3-70b", form="docs", docs=8, doc_len=1000, ragged=True),
        # One recomputed layer of a 20 % request over a 32k context, the query rows riding along:
        # what the headline request spends its time in.
        dict(name="layer_7b_32k", kind="layer", model="qwen2.5-7b", rows=6432, keys=32096),
        # The same in a mid-sized model and context, an odd number of rows.
        dict(name="layer_1.5b_16k", kind="layer", model="qwen2.5-1.5b", rows=3219, keys=16103),
        # One generated token over a long cache (server decoding), four layers and the lm_head.
        dict(name="decode_7b_32k", kind="append", model="qwen2.5-7b", layers=4, keys=32064, tokens=1),
        # A follow-up question of 32 tokens over the same cache: the query forward.
        dict(name="turn_7b_32k", kind="append", model="qwen2.5-7b", layers=4, keys=32064, tokens=32),
        # Plain reuse of four short cached documents in another order: the shortest whole request.
        dict(name="request_1k", kind="request", model="qwen2.5-0.5b", docs=4, doc_len=256, ragged=False, query=32,
             ratio=0.0, cold=False),
        # The request that the framework exists for: cached documents reordered, 20 % recomputed.
        dict(name="request_8k", kind="request", model="qwen2.5-0.5b", docs=8, doc_len=1000, ragged=False, query=32,
             ratio=0.2, cold=False),
        # A request none of whose documents is cached: hashed, packed, prefilled, stored or served.
        dict(name="request_cold_8k", kind="request", model="qwen2.5-0.5b", docs=8, doc_len=1000, ragged=True, query=32,
             ratio=0.0, cold=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """One more case of the ranges that the listed ones stand for."""
    kind = rng.choice(("assemble", "select", "attn", "attn", "layer", "layer", "append", "append", "append", "request"))
    small, mid, big, huge = "qwen2.5-0.5b", "qwen2.5-1.5b", "qwen2.5-7b", "llama3-70b"
    if kind == "assemble":
        model = rng.choice((small, mid, big))
        return dict(kind=kind, model=model, docs=rng.randint(1, 32), doc_len=_log_int(rng, 16, 1000), ragged=True)
    if kind == "select":
        return dict(kind=kind, model=rng.choice((small, mid, big, huge)), rows=_log_int(rng, 256, 32000),
                    ratio=rng.choice((0.05, 0.2, 0.5)))
    if kind == "attn":
        model = rng.choice((small, mid, big, huge))
        form = rng.choice(("causal", "docs", "rows"))
        if form == "causal":
            n = _log_int(rng, 64, 8096)
            return dict(kind=kind, model=model, form=form, rows=n, keys=n)
        if form == "docs":
            return dict(kind=kind, model=model, form=form, docs=rng.randint(1, 8), doc_len=_log_int(rng, 32, 1000),
                        ragged=True)
        keys = _log_int(rng, 512, 32096)
        return dict(kind=kind, model=model, form=form, rows=_log_int(rng, 2, max(2, keys // 5)), keys=keys)
    if kind == "layer":
        keys = _log_int(rng, 512, 32096)
        return dict(kind=kind, model=rng.choice((small, mid, big)), rows=_log_int(rng, 16, max(16, keys // 5)), keys=keys)
    if kind == "append":
        return dict(kind=kind, model=rng.choice((small, mid, big)), layers=rng.randint(2, 4),
                    keys=_log_int(rng, 256, 32064), tokens=rng.choice((1, 1, rng.randint(2, 8), rng.randint(9, 64))))
    return dict(kind=kind, model=small, docs=rng.randint(1, 8), doc_len=_log_int(rng, 32, 1000), ragged=True,
                query=rng.randint(1, 64), ratio=rng.choice((0.0, 0.2)), cold=rng.random() < 0.3)


# ------------------------------------------------------------------------------------- shared parts

def _cfg(case):
    cfg = preset(case["model"])
    if case["kind"] == "layer":  # one layer; its embedding is never read
        return cfg.scaled(num_hidden_layers=1, vocab_size=512)
    return cfg.scaled(num_hidden_layers=case["layers"]) if "layers" in case else cfg


def _doc_lens(case):
    """Lengths of a case's documents: equal, or between half and one and a half times the mean."""
    d, n = case["docs"], case["doc_len"]
    if not case["ragged"]:
        return [n] * d
    r = random.Random(1000 * d + n)
    return [max(1, round(n * r.uniform(0.5, 1.5))) for _ in range(d)]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, std=1.0):
    return torch.empty(shape, device="cuda", dtype=torch.bfloat16).normal_(0.0, std, generator=g)


def _ids(g, n, vocab):
    return torch.randint(0, vocab, (n,), generator=g, device="cuda")


def _model(case, seed):
    cfg = _cfg(case)
    return cfg, synthetic_model(cfg, "cuda", torch.bfloat16, seed=seed, std=0.02,
                                bias_std=0.05 if cfg.attention_bias else 0.0)


# Keys of twice the unit deviation against queries of about one: scores spread as in a trained
# model (a few hundred keys carry a row's weight), where unit keys would average all of V away.
KEY_STD = 2.0


def _attn_inputs(case, seed):
    """(q, K, V, kend, kseg or None, n_shared) of an attention case."""
    cfg, g = preset(case["model"]), _gen(seed)
    hq, hkv, hd = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
    kseg, n_shared = None, 0
    if case["form"] == "docs":
        lens = _doc_lens(case)
        n, n_shared = sum(lens), SYSTEM
        keys = n_shared + n
        kend = torch.arange(n_shared, keys, device="cuda")
        first = [n_shared + sum(lens[:i]) for i in range(len(lens))]
        kseg = torch.repeat_interleave(torch.tensor(first, device="cuda"), torch.tensor(lens, device="cuda"))
    else:
        n, keys = case["rows"], case["keys"]
        kend = torch.randperm(keys, generator=g, device="cuda")[:n].sort().values
    q = _randn(g, n, hq, hd)
    return q, _randn(g, 1, hkv, keys, hd, std=KEY_STD), _randn(g, 1, hkv, keys, hd), kend, kseg, n_shared


def _layer_inputs(case, seed):
    """(h [1, n, H], S, K, V): sorted recomputed positions, the last 32 rows (the query) among them."""
    cfg, g = _cfg(case), _gen(seed + 1)
    n, keys = case["rows"], case["keys"]
    tail = min(32, n // 2)
    S = torch.randperm(keys - tail, generator=g, device="cuda")[:n - tail].sort().values
    S = torch.cat([S, torch.arange(keys - tail, keys, device="cuda")])
    K = _randn(g, 1, cfg.num_key_value_heads, keys, cfg.head_dim, std=KEY_STD)
    return _randn(g, 1, n, cfg.hidden_size), S, K, _randn(g, 1, cfg.num_key_value_heads, keys, cfg.head_dim)


def _append_inputs(case, seed):
    """(ids, K, V): the tokens to append and the content of the cache before them."""
    cfg, g = _cfg(case), _gen(seed + 1)
    shape = (cfg.num_hidden_layers, 1, cfg.num_key_value_heads, case["keys"], cfg.head_dim)
    return _ids(g, case["tokens"], cfg.vocab_size), _randn(g, *shape, std=KEY_STD), _randn(g, *shape)


def _request_inputs(case, seed):
    """(system, docs, query, order): the documents as first seen and the request's order of them."""
    cfg, g = _cfg(case), _gen(seed + 1)
    system = _ids(g, SYSTEM, cfg.vocab_size)
    docs = [_ids(g, n, cfg.vocab_size) for n in _doc_lens(case)]
    order = list(range(len(docs)))
    random.Random(seed).shuffle(order)
    return system, docs, _ids(g, case["query"], cfg.vocab_size), order


def _select_inputs(case, seed):
    """(kv, cos, sin, rows, K, V, k): raw layer-1 k|v rows of every candidate and the cached layer.
    The cached rows are the fresh ones, rotated, with a drift that grows from candidate to candidate
    at random, as reordered documents have it."""
    cfg, g = preset(case["model"]), _gen(seed)
    n, hkv, hd = case["rows"], cfg.num_key_value_heads, cfg.head_dim
    kv = _randn(g, n, 2 * hkv * hd)
    rows = torch.arange(SYSTEM, SYSTEM + n, device="cuda")
    inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, hd, 2, dtype=torch.int64).float() / hd))
    ang = rows[:, None].float() * inv.to("cuda")[None]
    cos, sin = ang.cos().to(torch.bfloat16), ang.sin().to(torch.bfloat16)
    k = kv[:, :hkv * hd].reshape(n, hkv, hd).float()
    v = kv[:, hkv * hd:].reshape(n, hkv, hd).float()
    c, s = cos.float()[:, None], sin.float()[:, None]
    a, b = k[..., :hd // 2], k[..., hd // 2:]
    rot = torch.cat([a * c - b * s, b * c + a * s], dim=-1)
    drift = torch.rand(n, 1, 1, generator=g, device="cuda")
    K = _randn(g, 1, hkv, SYSTEM + n, hd)
    V = _randn(g, 1, hkv, SYSTEM + n, hd)
    noise = lambda: torch.randn(n, hkv, hd, generator=g, device="cuda") * drift
    K[0, :, SYSTEM:] = (rot + noise()).to(torch.bfloat16).transpose(0, 1)
    V[0, :, SYSTEM:] = (v + noise()).to(torch.bfloat16).transpose(0, 1)
    return kv, cos, sin, rows, K, V, int(round(case["ratio"] * n))


# ---------------------------------------------------------------------------------- prepare and run

def prepare(case, seed):
    with torch.inference_mode():
        return _prepare(case, seed)


def _prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "assemble":
        cfg, g = preset(case["model"]), _gen(seed)
        lens = [SYSTEM] + _doc_lens(case)
        shape = lambda n: (cfg.num_hidden_layers, 1, cfg.num_key_value_heads, n, cfg.head_dim)
        blocks = [(_randn(g, *shape(n)), _randn(g, *shape(n))) for n in lens]
        order = list(range(1, len(lens)))
        random.Random(seed).shuffle(order)
        src, off = [(*blocks[0], 0, 0)], SYSTEM
        for i in order:
            src.append((*blocks[i], off, off - SYSTEM))
            off += lens[i]
        inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, cfg.head_dim, 2, dtype=torch.int64).float() / cfg.head_dim))
        st.update(src=src, K=torch.zeros(shape(off), device="cuda", dtype=torch.bfloat16),
                  V=torch.zeros(shape(off), device="cuda", dtype=torch.bfloat16), inv=inv)
    elif kind == "select":
        st.update(inputs=_select_inputs(case, seed), cfg=preset(case["model"]))
    elif kind == "attn":
        st.update(inputs=_attn_inputs(case, seed), cfg=preset(case["model"]))
    elif kind == "layer":
        _, model = _model(case, seed)
        h, S, K, V = _layer_inputs(case, seed)
        # the row set's tables are built once and serve every layer of a recompute
        st.update(model=model, h=h, S=S, K=K, V=V, ctx=blend._subset_ctx(model, S, case["keys"], h))
    elif kind == "append":
        # the cache of a served request, replayed decoding on; its rows then hold this seed's content
        cfg, model = _model(case, seed)
        g = _gen(seed + 2)
        eng = Engine(model, BlockStore(1 << 20), graphs=True)
        T, q = case["keys"], 8
        _, cache, _ = eng.prefill(_ids(g, SYSTEM, cfg.vocab_size), [_ids(g, T - SYSTEM - q, cfg.vocab_size)],
                                  _ids(g, q, cfg.vocab_size), reserve=256)
        ids, K, V = _append_inputs(case, seed)
        cache.K[..., :T, :].copy_(K)
        cache.V[..., :T, :].copy_(V)
        st.update(eng=eng, cache=cache, ids=ids)
        eng.decode(cache, ids)  # the step's graph is captured on the first call of a size
    else:
        _, model = _model(case, seed)
        system, docs, query, order = _request_inputs(case, seed)
        # a store without room serves every block uncached: each pass is the first one on its documents
        eng = Engine(model, BlockStore(0 if case["cold"] else 1 << 33), graphs=True)
        if not case["cold"]:
            eng.prefill(system, docs, query)
        req = [docs[i] for i in order]
        eng.prefill(system, req[::-1], query, ratio=case["ratio"])  # the size's graphs are captured once
        st.update(eng=eng, system=system, docs=req, query=query)
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "assemble":
        _hip.rope_assemble(st["src"], st["K"], st["V"], st["inv"])
        return st["K"], st["V"]
    if kind == "select":
        kv, cos, sin, rows, K, V, k = st["inputs"]
        cfg = st["cfg"]
        score = _hip.dev_score(kv, cos, sin, rows, cfg.num_key_value_heads, cfg.head_dim, K, V)
        return score, _hip.topk_select(score, k)
    if kind == "attn":
        q, K, V, kend, kseg, n_shared = st["inputs"]
        cfg = st["cfg"]
        return _hip.subset_attn(q, K, V, kend, cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim,
                                cfg.head_dim ** -0.5, kseg=kseg, n_shared=n_shared)
    if kind == "layer":
        with torch.inference_mode():
            return blend._layer_subset(0, st["model"], st["h"], st["S"], st["K"], st["V"], inplace=True, ctx=st["ctx"])
    if kind == "append":
        cache = st["cache"]
        cache.length = case["keys"]  # the same position again
        logits = st["eng"].decode(cache, st["ids"])
        return logits, cache.K[..., :cache.length, :], cache.V[..., :cache.length, :]
    logits, cache, _ = st["eng"].prefill(st["system"], st["docs"], st["query"], ratio=case["ratio"])
    return logits, cache.K[..., :cache.length, :], cache.V[..., :cache.length, :]


# --------------------------------------------------------------------------------------------- work

def _layer_params(cfg):
    H, q, kv = cfg.hidden_size, cfg.num_attention_heads * cfg.head_dim, cfg.num_key_value_heads * cfg.head_dim
    return H * (q + 2 * kv) + q * H + 3 * H * cfg.intermediate_size


def _kv_row_bytes(cfg):
    """K and V bytes of one token in one layer."""
    return 2 * cfg.num_key_value_heads * cfg.head_dim * 2


def _attn_pairs(case):
    """(row, key) pairs of an attention case, per query head."""
    if case["form"] == "docs":
        return sum(n * SYSTEM + n * (n + 1) // 2 for n in _doc_lens(case))
    if case["form"] == "causal":
        return case["rows"] * (case["rows"] + 1) // 2
    return case["rows"] * (case["keys"] + 1) // 2


def work(case):
    """Bytes (inputs read once, outputs written once) and operations that one pass cannot do without."""
    kind, cfg = case["kind"], preset(case["model"])
    hq, hkv, hd, H = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim, cfg.hidden_size
    L = case.get("layers", cfg.num_hidden_layers)
    row = _kv_row_bytes(cfg)
    if kind == "assemble":
        T = SYSTEM + sum(_doc_lens(case))
        return {"bytes": 2 * T * cfg.num_hidden_layers * row, "flops": 3 * T * cfg.num_hidden_layers * hkv * hd}
    if kind == "select":
        n = case["rows"]
        return {"bytes": n * (2 * row + 2 * hd + 8 + 2) + 8 * int(round(case["ratio"] * n)), "flops": 8 * n * hkv * hd}
    if kind == "attn":
        n = sum(_doc_lens(case)) if case["form"] == "docs" else case["rows"]
        keys = SYSTEM + n if case["form"] == "docs" else case["keys"]
        return {"bytes": 2 * 2 * n * hq * hd + keys * row, "flops": 4 * hq * hd * _attn_pairs(case)}
    if kind == "layer":
        n, keys = case["rows"], case["keys"]
        return {"bytes": 2 * _layer_params(cfg) + 4 * n * H + (keys + n) * row,
                "flops": 2 * n * _layer_params(cfg) + 4 * hq * hd * n * (keys + 1) // 2}
    if kind == "append":
        n, T = case["tokens"], case["keys"]
        return {"bytes": 2 * (L * _layer_params(cfg) + cfg.vocab_size * H) + L * (T + 2 * n) * row,
                "flops": 2 * n * L * _layer_params(cfg) + 2 * cfg.vocab_size * H + 4 * hq * hd * L * n * (T + n // 2)}
    lens, nq = _doc_lens(case), case["query"]
    n, T = sum(lens), SYSTEM + sum(lens)
    rec = int(round(case["ratio"] * n))
    weights = 2 * (L * _layer_params(cfg) + cfg.vocab_size * H)
    flops = 2 * nq * L * _layer_params(cfg) + 2 * cfg.vocab_size * H + 4 * hq * hd * L * nq * T
    if rec:  # layer 0 of every row, the other layers of the recomputed ones
        flops += 2 * n * _layer_params(cfg) + 2 * hq * hd * T * T
        flops += (L - 1) * (2 * rec * _layer_params(cfg) + 2 * hq * hd * rec * T)
    if case["cold"]:
        flops += L * (2 * T * _layer_params(cfg) + 4 * hq * hd * (SYSTEM * SYSTEM // 2 + sum(
            m * SYSTEM + m * (m + 1) // 2 for m in lens)))
    # weights, the assembled cache written once, its blocks read once, the cache read by the query
    return {"bytes": weights + 3 * T * L * row, "flops": flops}


# ----------------------------------------------------------------------------------------- tolerance

def tolerance(case):
    """Largest relative error (2-norm over 2-norm, every output) of another correct implementation."""
    kind = case["kind"]
    if kind in ("assemble", "select"):
        # fixed fp32 operations on each element and one rounding; the selection's ties go to the
        # lowest index: nothing is left to an implementation
        return "exact"
    # About four times the distance measured between run and exact (attention 3.5e-3, a layer 5.5e-3:
    # bf16 inputs to every product, one rounding of each result), and for the logits of several bf16
    # layers about three times (1.5e-2 to 2.3e-2 from exact; 1.7e-2 between two orders of the same
    # request's sums). The caches that come back with them are much closer.
    return {"rel": {"attn": 1.2e-2, "layer": 2e-2, "append": 6e-2, "request": 6e-2}[kind]}


# -------------------------------------------------------------------------------------------- exact

def _rope64(x, pos, inv):
    """Rotate x [n, heads, hd] by the positions pos [n], split-half convention."""
    ang = pos.double()[:, None] * inv.double()[None].to(x.device)
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x.chunk(2, dim=-1)
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _attn64(q, K, V, kend, kseg=None, n_shared=0):
    """q [n, hq, hd], K, V [hkv, T, hd] in 64 bits; row i sees keys <= kend[i] outside
    [n_shared, kseg[i])."""
    n, hq, hd = q.shape
    hkv, T = K.shape[0], K.shape[1]
    G = hq // hkv
    out = torch.empty_like(q)
    key = torch.arange(T, device=q.device)
    step = max(1, (1 << 28) // (T * G * 8))
    for i in range(0, n, step):
        e = kend[i:i + step, None]
        see = key[None] <= e
        if kseg is not None:
            see &= (key[None] < n_shared) | (key[None] >= kseg[i:i + step, None])
        for h in range(hkv):
            x = q[i:i + step, h * G:(h + 1) * G].reshape(-1, hd)
            s = (x @ K[h].t().contiguous()) * hd ** -0.5
            s = s.view(-1, G, T).masked_fill_(~see[:, None], -math.inf).softmax(dim=-1)
            out[i:i + step, h * G:(h + 1) * G] = (s.view(-1, T) @ V[h]).view(-1, G, hd)
    return out


def _norm64(x, w, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w.double()


def _linear64(x, lin):
    y = x @ lin.weight.double().t().contiguous()
    return y if lin.bias is None else y + lin.bias.double()


def _layer64(cfg, layer, inv, h, pos, rows, kend, K, V, kseg=None, n_shared=0):
    """One decoder layer of rows h [n, H] in 64 bits; K, V [hkv, T, hd] take their k and v."""
    n, hd = h.shape[0], cfg.head_dim
    at = layer.self_attn
    x = _norm64(h, layer.input_layernorm.weight, cfg.rms_norm_eps)
    q = _rope64(_linear64(x, at.q_proj).view(n, -1, hd), pos, inv)
    K[:, rows] = _rope64(_linear64(x, at.k_proj).view(n, -1, hd), pos, inv).transpose(0, 1)
    V[:, rows] = _linear64(x, at.v_proj).view(n, -1, hd).transpose(0, 1)
    h = h + _linear64(_attn64(q, K, V, kend, kseg, n_shared).reshape(n, -1), at.o_proj)
    x = _norm64(h, layer.post_attention_layernorm.weight, cfg.rms_norm_eps)
    g = _linear64(x, layer.mlp.gate_proj)
    return h + _linear64(g * torch.sigmoid(g) * _linear64(x, layer.mlp.up_proj), layer.mlp.down_proj)


def _forward64(cfg, model, ids, K, V, rows, pos=None, kseg=None, n_shared=0):
    """Every layer for token ids at cache rows `rows` (positions pos), K, V [L, hkv, T, hd]."""
    inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, cfg.head_dim, 2, dtype=torch.int64).float() / cfg.head_dim))
    h = model.model.embed_tokens.weight[ids].double()
    for l, layer in enumerate(model.model.layers):
        h = _layer64(cfg, layer, inv, h, rows if pos is None else pos, rows, rows, K[l], V[l], kseg, n_shared)
    return h


def _logits64(cfg, model, h):
    return _linear64(_norm64(h[-1:], model.model.norm.weight, cfg.rms_norm_eps), model.lm_head)[0]


def exact(case, seed):
    """run's outputs in 64 bits from the same inputs."""
    with torch.inference_mode():
        return _exact(case, seed)


def _exact(case, seed):
    kind = case["kind"]
    if kind == "assemble":
        st = _prepare(case, seed)
        K, V = torch.empty_like(st["K"], dtype=torch.float64), torch.empty_like(st["V"], dtype=torch.float64)
        for k, v, off, delta in st["src"]:
            n, hd = k.shape[-2], k.shape[-1]
            flat = k.double().reshape(-1, 1, hd)
            shift = torch.full((flat.shape[0],), delta, device="cuda")
            K[..., off:off + n, :] = _rope64(flat, shift, st["inv"]).view(k.shape)
            V[..., off:off + n, :] = v.double()
        return K, V
    if kind == "select":
        kv, cos, sin, rows, K, V, _ = _select_inputs(case, seed)
        cfg = preset(case["model"])
        n, hkv, hd = kv.shape[0], cfg.num_key_value_heads, cfg.head_dim
        k, v = kv.double().view(n, 2, hkv, hd).unbind(1)
        a, b = k.chunk(2, dim=-1)
        c, s = cos.double()[:, None], sin.double()[:, None]
        dk = torch.cat([a * c - b * s, b * c + a * s], dim=-1) - K[0][:, rows].double().transpose(0, 1)
        dv = v - V[0][:, rows].double().transpose(0, 1)
        return dk.norm(dim=-1).sum(-1) + dv.norm(dim=-1).sum(-1), None  # ties make the indices
    if kind == "attn":
        q, K, V, kend, kseg, n_shared = _attn_inputs(case, seed)
        return _attn64(q.double(), K[0].double(), V[0].double(), kend, kseg, n_shared).reshape(q.shape[0], -1)
    if kind == "layer":
        cfg, model = _model(case, seed)
        h, S, K, V = _layer_inputs(case, seed)
        inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, cfg.head_dim, 2, dtype=torch.int64).float() / cfg.head_dim))
        K, V = K.double(), V.double()
        return _layer64(cfg, model.model.layers[0], inv, h[0].double(), S, S, S, K[0], V[0])[None], K, V
    cfg, model = _model(case, seed)
    L, hkv, hd = cfg.num_hidden_layers, cfg.num_key_value_heads, cfg.head_dim
    room = lambda n: torch.zeros(L, hkv, n, hd, device="cuda", dtype=torch.float64)
    if kind == "append":
        ids, K0, V0 = _append_inputs(case, seed)
        T, n = case["keys"], case["tokens"]
        K, V = room(T + n), room(T + n)
        K[:, :, :T], V[:, :, :T] = K0[:, 0], V0[:, 0]
        h = _forward64(cfg, model, ids, K, V, torch.arange(T, T + n, device="cuda"))
        return _logits64(cfg, model, h), K[:, None], V[:, None]
    if case["ratio"] > 0:
        return None  # which rows tie at the selection's threshold has no 64-bit answer
    system, docs, query, order = _request_inputs(case, seed)
    P, T, nq = SYSTEM, SYSTEM + sum(map(len, docs)), len(query)
    K, V = room(T + nq), room(T + nq)
    Kp, Vp = room(P), room(P)
    _forward64(cfg, model, system, Kp, Vp, torch.arange(P, device="cuda"))
    K[:, :, :P], V[:, :, :P] = Kp, Vp
    inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, hd, 2, dtype=torch.int64).float() / hd))
    off = P
    for i in order:  # each document on top of the system prompt, moved to its place
        n = len(docs[i])
        Kd, Vd = room(P + n), room(P + n)
        Kd[:, :, :P], Vd[:, :, :P] = Kp, Vp
        _forward64(cfg, model, docs[i], Kd, Vd, torch.arange(P, P + n, device="cuda"))
        flat = Kd[:, :, P:].reshape(-1, 1, hd)
        shift = torch.full((flat.shape[0],), off - P, device="cuda")
        K[:, :, off:off + n] = _rope64(flat, shift, inv).view(L, hkv, n, hd)
        V[:, :, off:off + n] = Vd[:, :, P:]
        off += n
    h = _forward64(cfg, model, query, K, V, torch.arange(T, T + nq, device="cuda"))
    return _logits64(cfg, model, h), K[:, None], V[:, None]
