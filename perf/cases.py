"""Performance cases of the paged INT4 / fp16 KV-cache data plane.

A case is one call (or the short sequence of calls) that a serving program
makes per layer, through ``memopt_C`` and ``memopt_runtime``:

* ``attend``: ``dynamic_sparse_attention`` (or the ``PreparedAttention`` a
  decode loop keeps) over INT4 pages (``layout="pages"``), the reference's
  token-major INT4 codes (``"rows"``) or an fp16 pool (``"fp16"``); decode
  (``q_len`` 1), a few tokens per sequence, chunks, whole prompts;
* ``step``: one decode step on the live pool, ``write_cache`` of the new
  token of every sequence, then attention;
* ``autochunk``: ``autochunk_prefill`` of one prompt on a ``PagedKVCache``;
* ``compress``: a prompt's K/V written into the live INT4 pool and thinned
  with ``evict_tokens``;
* ``quant``: the surface ``quantize_kv_cache_int4`` of a pool tensor and
  ``dequantize_kv_cache_int4`` of the result.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "memopt-transformer-runtime_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import memopt_C  # noqa: E402
import memopt_runtime  # noqa: E402

DEV = "cuda"


def _attend(**kw):
    case = dict(kind="attend", layout="pages", batch=1, heads=32, dim=128, block=16, ctx=4096, q_len=1, window=-1,
                sinks=4, causal=False, ragged=False, holes=False, std=1.0, plan=False)
    case.update(kw)
    return case


def listed():
    return [
        # The smallest decode of the repository's configurations: one sequence of 1024 tokens, 8 heads of 64,
        # over the codes and fp32 scales that quantize_kv_cache_int4 returns. Latency and launches.
        _attend(name="decode_rows_small", layout="rows", heads=8, dim=64, ctx=1024),
        # The headline decode: 16 sequences of 4096 tokens, 32 heads of 128, INT4 pages, a kept plan.
        _attend(name="decode_pages_batch", batch=16, ctx=4096, plan=True),
        # Sparse decode of a served batch: unequal contexts up to 8192, a 2048-token window, sinks, and block
        # tables with the holes that eviction leaves.
        _attend(name="decode_pages_window", batch=16, ctx=8192, window=2048, ragged=True, holes=True, plan=True),
        # One user's long context: a single sequence of 131072 tokens.
        _attend(name="decode_pages_long", ctx=131072),
        # A decode step in the default (fp16) cache: 8 sequences of unequal length, the new tokens' K/V written
        # into the live pool, then attention over it.
        dict(name="step_fp16", kind="step", layout="fp16", batch=8, heads=32, dim=128, ctx=4000, ragged=True,
             window=-1, sinks=0),
        # A few tokens per sequence at once (PolicyForward.step with T new tokens): 5 queries on 8 sequences.
        _attend(name="few_queries_pages", batch=8, ctx=4000, q_len=5, causal=True, ragged=True),
        # A 5000-token prompt prefilled in chunks of 512 under a 1024-token window, INT4 pages.
        dict(name="autochunk_pages", kind="autochunk", heads=32, dim=128, ctx=5000, chunk=512, window=1024, sinks=4),
        # One-shot prefill of a long prompt: 16384 tokens, window 4096, 4 sinks, INT4 pages.
        _attend(name="prefill_pages_long", ctx=16384, q_len=16384, window=4096, causal=True, std=0.5),
        # The reference's own attention call: DynamicAttention over the fp16 pool, non-causal, full window, every
        # position a query (2 sequences, 8 heads of 64).
        _attend(name="attend_fp16_full", layout="fp16", batch=2, heads=8, dim=64, ctx=1024, q_len=1024, window=1024,
                sinks=0),
        # Several queries over token-major INT4 codes: the reference's INT4 cache on a chunk of a prompt.
        _attend(name="attend_rows_chunk", layout="rows", batch=2, heads=8, dim=64, ctx=1024, q_len=100),
        # Surface quantize of a pool tensor and back.
        dict(name="quant_roundtrip", kind="quant", pages=2039, heads=32, dim=128),
        # Four prompts of 6005 tokens written into the INT4 pool and thinned to three quarters.
        dict(name="compress_pages", kind="compress", batch=4, heads=32, dim=128, ctx=6005, retain=0.75, sinks=4),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "few", "chunk", "prefill", "full", "step", "autochunk", "quant",
                       "compress"])
    heads, dim = rng.choice([(8, 64), (12, 64), (8, 128), (32, 128), (32, 128), (20, 64), (40, 128)])
    window = rng.choice([-1, -1, 512, 1024, 2048, 4096])
    sinks = rng.choice([0, 4, 4, 16])
    if kind == "decode":
        batch = _log_int(rng, 1, 32)
        layout = rng.choice(["pages", "pages", "rows", "fp16"])
        most = 2 ** 21 // (batch * heads * dim // 128)  # at most 2^21 (token, head) rows of 128 dims per batch entry
        return _attend(layout=layout, batch=batch, heads=heads, dim=dim, ctx=_log_int(rng, 64, min(131072, most)),
                       block=rng.choice([16, 16, 32]) if layout == "fp16" else 16, window=window, sinks=sinks,
                       ragged=rng.random() < 0.5, holes=rng.random() < 0.3, plan=rng.random() < 0.3)
    if kind in ("few", "chunk"):
        q_len = _log_int(rng, 2, 16) if kind == "few" else _log_int(rng, 17, 1024)
        batch = _log_int(rng, 1, 16) if kind == "few" else rng.choice([1, 1, 2, 4])
        layout = rng.choice(["pages", "pages", "fp16", "rows"])
        # token-major codes with several queries: at the sizes of that cache's own configuration
        ctx = _log_int(rng, 256, 2048) if layout == "rows" else _log_int(rng, 512, 32768 // batch)
        if layout == "rows":
            heads, dim, q_len = 8, 64, min(q_len, 256)
        return _attend(layout=layout, batch=batch, heads=heads, dim=dim, ctx=max(ctx, 2 * q_len), q_len=q_len,
                       window=window, sinks=sinks, causal=True, ragged=batch > 1 and rng.random() < 0.5)
    if kind == "prefill":
        ctx = _log_int(rng, 300, 16384)
        return _attend(layout=rng.choice(["pages", "pages", "fp16"]), heads=min(heads, 32), dim=dim, ctx=ctx,
                       q_len=ctx, window=window if window > 0 else min(ctx, 4096), sinks=sinks, causal=True, std=0.5)
    if kind == "full":
        ctx = _log_int(rng, 100, 2048)
        return _attend(layout="fp16", batch=rng.choice([1, 2, 4]), heads=heads, dim=dim, ctx=ctx, q_len=ctx,
                       block=rng.choice([16, 32]), window=rng.choice([ctx, max(16, ctx // 2)]), sinks=0)
    if kind == "step":
        batch = _log_int(rng, 1, 32)
        return dict(kind="step", layout=rng.choice(["fp16", "pages", "pages"]), batch=batch, heads=heads, dim=dim,
                    ctx=_log_int(rng, 100, 65536 // batch), ragged=rng.random() < 0.7, window=window, sinks=sinks)
    if kind == "autochunk":
        return dict(kind="autochunk", heads=heads, dim=dim, ctx=_log_int(rng, 500, 10000),
                    chunk=rng.choice([128, 300, 512, 1000, 2048]), window=window if window > 0 else 4096, sinks=sinks)
    if kind == "quant":
        return dict(kind="quant", pages=_log_int(rng, 3, 4096), heads=heads, dim=dim)
    return dict(kind="compress", batch=rng.choice([1, 2, 4, 8]), heads=heads, dim=dim,
                ctx=_log_int(rng, 500, 8192), retain=rng.choice([0.5, 0.75, 0.9]), sinks=sinks)


# ---------------------------------------------------------------------------
# Inputs (from the seed alone)
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _kv(shape, g, std=1.0):
    """fp16 keys or values: normal, with the 1 % of outliers (x8) that quantization groups meet."""
    x = torch.randn(shape, generator=g, device=DEV, dtype=torch.float16)
    if std != 1.0:
        return x.mul_(std)
    return x.mul_(torch.rand(shape, generator=g, device=DEV, dtype=torch.float16).lt_(0.01).mul_(7.0).add_(1.0))


def _lens(case):
    """Context lengths; ragged ones lie between ctx / 3 and ctx, and hold the queries."""
    n, ctx = case["batch"], case["ctx"]
    if not case["ragged"]:
        return [ctx] * n
    return [max(case.get("q_len", 1), ctx - (i * 977 + 13) % max(1, 2 * ctx // 3) if i else ctx) for i in range(n)]


def _tables(case, pages_per_seq, g):
    """A random permutation of the page pool dealt to the sequences, int32 [B, M]."""
    bt = torch.randperm(case["batch"] * pages_per_seq, generator=g, device=DEV).to(torch.int32)
    bt = bt.view(case["batch"], pages_per_seq)
    if case.get("holes"):  # pages that eviction unlinked
        bt[:, 2::23] = -1
    return bt.contiguous()


def _attend_inputs(case, seed):
    g = _gen(seed)
    B, H, D, bs = case["batch"], case["heads"], case["dim"], case["block"]
    m = -(-case["ctx"] // bs)
    k = _kv((B * m, bs, H, D), g, case["std"])
    v = _kv((B * m, bs, H, D), g, case["std"])
    q = torch.randn((B, case["q_len"], H, D), generator=g, device=DEV, dtype=torch.float16).mul_(case["std"])
    lens = _lens(case)
    return q, k, v, _tables(case, m, g), lens, torch.tensor(lens, dtype=torch.int32, device=DEV)


def _token_slots(bt, starts, count, bs):
    """int32 slots of `count` positions from starts[i] of every sequence, sequence-major."""
    pos = starts[:, None] + torch.arange(count, device=DEV)
    page = torch.gather(bt.long(), 1, pos // bs)
    return (page * bs + pos % bs).to(torch.int32).flatten().contiguous()


def _step_inputs(case, seed):
    """The live pool's contents and tables belong to the case (one pool serves every state of it); the seed
    makes the step's query and new keys and values."""
    g0 = _gen(977)
    B, H, D = case["batch"], case["heads"], case["dim"]
    m = -(-case["ctx"] // 16)
    k, v = _kv((B * m * 16, H, D), g0), _kv((B * m * 16, H, D), g0)
    bt = _tables(case, m, g0)
    lens = _lens(case)
    ctx = torch.tensor(lens, dtype=torch.int32, device=DEV)
    slots = _token_slots(bt, ctx.long() - 1, 1, 16)
    g = _gen(seed)
    q = torch.randn((B, 1, H, D), generator=g, device=DEV, dtype=torch.float16)
    return q, k, v, _kv((B, H, D), g), _kv((B, H, D), g), bt, lens, ctx, slots


def _prompt_inputs(case, seed):
    g = _gen(seed)
    S, H, D = case["ctx"], case["heads"], case["dim"]
    q = torch.randn((S, H, D), generator=g, device=DEV, dtype=torch.float16)
    return q, _kv((S, H, D), g), _kv((S, H, D), g)


_engine = {}


def _fresh_pool(pages, heads, dim, fmt):
    _engine.clear()
    memopt_C.reset_pool()
    memopt_C.init_pool(pages, 16, heads, dim, kv_format=fmt)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "attend":
        q, k, v, bt, lens, ctx = _attend_inputs(case, seed)
        st = dict(case=case, q=q, bt=bt, ctx=ctx, max_len=max(lens), scales={})
        if case["layout"] == "fp16":
            st["k"], st["v"] = k, v
        elif case["layout"] == "rows":
            st["k"], ks = memopt_C.quantize_kv_cache_int4(k, 64)
            st["v"], vs = memopt_C.quantize_kv_cache_int4(v, 64)
            st["scales"] = dict(key_scales=ks, value_scales=vs, kv_layout="token_major")
        else:
            nb, H, D = k.shape[0], case["heads"], case["dim"]
            _fresh_pool(nb, H, D, "int4")
            memopt_C.write_cache(k.view(-1, H, D), v.view(-1, H, D), bt,
                                 torch.arange(nb * 16, dtype=torch.int32, device=DEV), validate_slots=False)
            st["k"] = st["v"] = memopt_C.get_int4_pages()
            memopt_C.reset_pool()
        if case["plan"]:
            st["plan"] = memopt_C.PreparedAttention(q, st["k"], st["v"], bt, ctx, st["max_len"], case["window"],
                                                    num_sink_tokens=case["sinks"], causal=case["causal"],
                                                    **st["scales"])
        return st
    if kind == "step":
        q, k, v, nk, nv, bt, lens, ctx, slots = _step_inputs(case, seed)
        _engine.clear()
        memopt_C.init_pool(bt.numel(), 16, case["heads"], case["dim"],
                           kv_format="fp16" if case["layout"] == "fp16" else "int4")
        memopt_C.write_cache(k, v, bt, torch.arange(bt.numel() * 16, dtype=torch.int32, device=DEV),
                             validate_slots=False)
        return dict(case=case, q=q, k=nk, v=nv, bt=bt, ctx=ctx, max_len=max(lens), slots=slots)
    if kind == "autochunk":
        q, k, v = _prompt_inputs(case, seed)
        key = (case["ctx"], case["heads"], case["dim"])
        if _engine.get("key") != key:  # one cache serves every prompt of the case
            pages = -(-case["ctx"] // 16)
            _engine.clear()
            _engine.update(key=key, cache=memopt_runtime.PagedKVCache(2 * pages + 7, case["heads"], case["dim"],
                                                                      kv_format="int4"))
        return dict(case=case, q=q, k=k, v=v, cache=_engine["cache"])
    if kind == "quant":
        return dict(case=case, x=_kv((case["pages"], 16, case["heads"], case["dim"]), _gen(seed)))
    # compress: every pass writes every row of the live pool before it evicts
    g = _gen(seed)
    N, H, D, L = case["batch"], case["heads"], case["dim"], case["ctx"]
    m = -(-L // 16)
    bt = _tables(case, m, _gen(977))
    slots = _token_slots(bt, torch.zeros(N, dtype=torch.long, device=DEV), L, 16)
    _fresh_pool(N * m, H, D, "int4")
    return dict(case=case, k=_kv((N * L, H, D), g), v=_kv((N * L, H, D), g), bt=bt, slots=slots,
                scores=torch.randn((N, H, L), generator=g, device=DEV).exp_())


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "attend":
        if "plan" in st:
            return st["plan"]()
        return memopt_C.dynamic_sparse_attention(st["q"], st["k"], st["v"], st["bt"], st["ctx"], st["max_len"],
                                                 case["window"], num_sink_tokens=case["sinks"],
                                                 causal=case["causal"], **st["scales"])
    if kind == "step":
        memopt_C.write_cache(st["k"], st["v"], st["bt"], st["slots"], validate_slots=False)
        k, v = memopt_C.get_key_pool(), memopt_C.get_value_pool()
        out = memopt_C.dynamic_sparse_attention(st["q"], k, v, st["bt"], st["ctx"], st["max_len"], case["window"],
                                                num_sink_tokens=case["sinks"])
        return [out, k, v] if case["layout"] == "fp16" else [out, memopt_C.get_int4_pages()]
    if kind == "autochunk":
        cache = st["cache"]
        cache.add_sequence(0)
        out = memopt_runtime.autochunk_prefill(cache, 0, st["q"], st["k"], st["v"], window_size=case["window"],
                                               num_sink_tokens=case["sinks"], chunk_tokens=case["chunk"])
        cache.free_sequence(0)
        return out
    if kind == "quant":
        packed, scales = memopt_C.quantize_kv_cache_int4(st["x"], 64)
        return [packed, scales, memopt_C.dequantize_kv_cache_int4(packed, scales, 64)]
    bt = st["bt"].clone()  # unlinked in place by the eviction
    votes = torch.zeros(bt.numel(), dtype=torch.int32, device=DEV)
    memopt_C.write_cache(st["k"], st["v"], bt, st["slots"], validate_slots=False)
    memopt_C.evict_tokens(st["scores"], bt, votes, case["retain"], case["sinks"])
    return [memopt_C.get_int4_pages(), bt, votes]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def _kv_bytes(layout, dim):
    """Stored bytes of one (token, head) of K and V."""
    if layout == "fp16":
        return 4 * dim
    return 2 * (dim // 2 + (dim // 64) * (2 if layout == "pages" else 4))


def _visible(ctx, q_len, window, max_len, sinks, causal):
    """(keys that some query sees, (query, key) pairs) of one sequence and head."""
    w = max_len if window <= 0 or window > max_len else window
    s = min(sinks, ctx)
    if not causal:
        n = min(ctx, min(ctx, w) + min(s, max(0, ctx - w)))
        return n, n * q_len
    pairs = 0
    for pos in range(ctx - q_len, ctx):
        lo = max(0, pos - w + 1)
        pairs += pos + 1 - lo + min(s, lo)
    lo = max(0, ctx - q_len - w + 1)
    return ctx - lo + min(s, lo), pairs


def work(case):
    kind = case["kind"]
    H, D = case["heads"], case["dim"]
    if kind in ("attend", "step"):
        lens = _lens(case)
        q_len, causal = case.get("q_len", 1), case.get("causal", False)
        seen = [_visible(n, q_len, case["window"], max(lens), case["sinks"], causal) for n in lens]
        share = 22 / 23 if case.get("holes") else 1.0
        keys, pairs = share * sum(s[0] for s in seen), share * sum(s[1] for s in seen)
        rows = len(lens) * q_len * H * D * 2
        new = len(lens) * H * (4 * D + _kv_bytes(case["layout"], D)) if kind == "step" else 0
        return {"bytes": keys * H * _kv_bytes(case["layout"], D) + 2 * rows + new, "flops": 4.0 * pairs * H * D}
    if kind == "autochunk":
        S = case["ctx"]
        _, pairs = _visible(S, S, case["window"], S, case["sinks"], True)
        return {"bytes": S * H * (2 * 2 * D + 4 * D + 2 * _kv_bytes("pages", D)), "flops": 4.0 * pairs * H * D}
    if kind == "quant":
        n = case["pages"] * 16 * H * D
        return {"bytes": n * (2 + 0.5 + 4 / 64) + n * (0.5 + 4 / 64 + 2), "flops": 0}
    n = case["batch"] * case["ctx"] * H
    return {"bytes": n * (4 * D + _kv_bytes("pages", D) + 4), "flops": 0}


def tolerance(case):
    if case["kind"] in ("quant", "compress"):
        return "exact"
    # Outputs are fp16 (2^-11 of a value, 2e-4 in the 2-norm) and probabilities meet V as fp16 in the matrix
    # products: 2.1e-4 to 2.5e-4 against 64 bits. The one-query INT4 path multiplies code and scale without rounding
    # the product to fp16 as the stated round trip does: 6e-4 (1024 tokens) to 1.2e-3 (131072 tokens).
    one_query = case["kind"] == "step" or case.get("q_len") == 1
    return {"rel": 4e-3 if one_query and case["layout"] != "fp16" else 1e-3}


# ---------------------------------------------------------------------------
# The same results in 64 bits
# ---------------------------------------------------------------------------

def _restored(x, page_scales=True):
    """Group-64 INT4 round trip of fp16 x: what the cache holds of it, as dequantize_kv_cache_int4 states it."""
    out = torch.empty_like(x)
    for src, dst in zip(x.view(-1, 64).split(1 << 22), out.view(-1, 64).split(1 << 22)):
        f = src.double()  # the scale and the quotient are those of an IEEE division in 32 bits
        amax = f.abs().amax(1, keepdim=True)
        scale = torch.where(amax > 0, amax / 7, torch.ones_like(amax)).float()
        q = (f / scale.double()).float().double()
        code = torch.sign(q) * torch.floor(q.abs() + 0.5)
        if page_scales:
            scale = scale.half()
            scale = torch.where(scale == 9360, torch.full_like(scale, 9352), scale)
        dst.copy_((code * scale.double()).half())
    return out


def _attention64(q, k, v, bt, lens, block, window, sinks, causal):
    B, Lq, H, D = q.shape
    out = torch.zeros(q.shape, dtype=torch.float64, device=DEV)
    most = max(lens)
    w = most if window <= 0 or window > most else window
    for b in range(B):
        n = lens[b]
        pages = bt[b, : -(-n // block)].long()
        key = torch.arange(n, device=DEV)
        linked = (pages >= 0).repeat_interleave(block)[:n]
        if not causal:
            use = linked & ((key >= n - w) | (key < sinks))
            key, linked = key[use], linked[use]
        slot = pages.clamp(min=0)[key // block] * block + key % block
        for h in range(H):
            kk = k.view(-1, H, D)[slot, h].double()
            vv = v.view(-1, H, D)[slot, h].double()
            for i in range(0, Lq, 2048):
                s = q[b, i:i + 2048, h].double() @ kk.T / math.sqrt(D)
                if causal:
                    pos = n - Lq + torch.arange(i, min(Lq, i + 2048), device=DEV)[:, None]
                    s.masked_fill_(~(linked & (key <= pos) & ((key < sinks) | (key >= pos - w + 1))), -math.inf)
                out[b, i:i + 2048, h] = torch.softmax(s, 1).nan_to_num_(0.0) @ vv
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "attend":
        q, k, v, bt, lens, _ = _attend_inputs(case, seed)
        if case["layout"] != "fp16":
            k, v = (_restored(x, case["layout"] == "pages") for x in (k, v))
        return _attention64(q, k, v, bt, lens, case["block"], case["window"], case["sinks"], case["causal"])
    if kind == "step":
        q, k, v, nk, nv, bt, lens, _, slots = _step_inputs(case, seed)
        k[slots.long()], v[slots.long()] = nk, nv
        pools = [None, None]
        if case["layout"] != "fp16":
            k, v, pools = _restored(k), _restored(v), [None]
        return [_attention64(q, k, v, bt, lens, 16, case["window"], case["sinks"], False)] + pools
    if kind == "autochunk":
        q, k, v = _prompt_inputs(case, seed)
        bt = torch.arange(-(-case["ctx"] // 16), device=DEV)[None]
        return _attention64(q[None], _restored(k), _restored(v), bt, [case["ctx"]], 16, case["window"],
                            case["sinks"], True)[0]
    if kind == "quant":
        x = prepare(case, seed)["x"].double()
        amax = x.view(-1, 64).abs().amax(1)
        return [None, torch.where(amax > 0, amax / 7, torch.ones_like(amax)), None]
    return None
