"""The attention passes that a serving program has this package do, as measurable cases.

Every case is one pass of the attention layers of a model through the vLLM backend classes:
``TTAttentionBackendImpl.forward`` (decode step, first prefill chunk, continuation chunk) or
``TTMLAAttentionBackendImpl.forward`` (the latent layers).  What a serving program has at hand
before that call is made by ``prepare``: the backend object of a layer, its paged caches, the
metadata of the pass from ``PagedMetadataBuilder``, the activations and the output buffer; and,
where ``graph`` is set, the captured decode forward (decode passes of a serving loop are replayed
from a HIP graph; prefill passes change their shape from pass to pass and run eagerly).

Contexts of a batch are spread evenly over the logarithm of [ctx_lo, ctx_hi] and shuffled by the
seed, so the work of a case does not depend on the seed.
"""

import math
import os
import sys
import types

import numpy as np
import torch

_PACKAGE_ROOT = os.path.abspath("tt-xla_amd")
if _PACKAGE_ROOT not in sys.path:
    sys.path.insert(0, _PACKAGE_ROOT)

# (query heads, KV heads, head size) of the layers: the shapes of the benchmark and of the tests
_HEADS = [(8, 8, 64), (8, 2, 64), (64, 8, 64), (16, 16, 128), (16, 8, 128), (32, 8, 128), (40, 8, 128),
          (64, 8, 128), (16, 8, 256)]
# latent layers: features of the no-position and the rotary part of a head, latent width, value width
_NOPE, _ROPE, _LATENT, _VHEAD = 128, 64, 512, 128

# a drawn case costs no more than the largest listed ones
_MAX_BYTES, _MAX_FLOPS = 3.3e9, 2.9e11


def _decode(users, heads, block, ctx_lo, ctx_hi, layers=1, graph=False, bfp8=False, window=0, sinks=False, parked=0):
    hq, hkv, d = heads
    return {"kind": "decode", "users": users, "q_heads": hq, "kv_heads": hkv, "head_size": d, "block": block,
            "ctx_lo": ctx_lo, "ctx_hi": ctx_hi, "layers": layers, "graph": graph, "bfp8": bfp8, "window": window,
            "sinks": sinks, "parked": parked}


def _prefill(users, tokens, heads, block, start=0, bfp8=False, window=0):
    hq, hkv, d = heads
    return {"kind": "prefill", "users": users, "tokens": tokens, "q_heads": hq, "kv_heads": hkv, "head_size": d,
            "block": block, "start": start, "bfp8": bfp8, "window": window}


def _latent_decode(users, heads, block, ctx_lo, ctx_hi):
    return {"kind": "latent-decode", "users": users, "q_heads": heads, "block": block, "ctx_lo": ctx_lo, "ctx_hi": ctx_hi}


def _latent_prefill(users, tokens, heads, block):
    return {"kind": "latent-prefill", "users": users, "tokens": tokens, "q_heads": heads, "block": block}


def listed():
    small, l8b, l70b, narrow = (8, 8, 64), (32, 8, 128), (64, 8, 128), (64, 8, 64)
    return [
        # one request, short context, no graph: what a single user waits for per layer and token
        dict(_decode(1, small, 32, 128, 128), name="decode-one"),
        # an ordinary serving batch of an 8B model: four layers of a captured decode forward
        dict(_decode(32, l8b, 64, 512, 4096, layers=4, graph=True), name="decode-batch"),
        # the same batch with the block-float-8 cache option; five rows of the bucket are parked
        dict(_decode(32, l8b, 64, 512, 4096, layers=4, graph=True, bfp8=True, parked=5), name="decode-bfp8"),
        # a full batch of a 70B model with very ragged contexts: the largest decode pass
        dict(_decode(128, l70b, 64, 256, 32768), name="decode-long"),
        # sliding-window layers with sinks at the page size that the backend asks for (32)
        dict(_decode(37, narrow, 32, 1024, 32768, layers=4, graph=True, window=1024, sinks=True), name="decode-window"),
        # a short prompt of one request (its token bucket): time to the first token
        dict(_prefill(1, 128, l8b, 32), name="prefill-short"),
        # ordinary prompts, first chunk: cache fill and dense causal attention
        dict(_prefill(4, 2048, l8b, 64), name="prefill-first"),
        # long prompts on sliding-window layers
        dict(_prefill(2, 4096, l8b, 32, window=1024), name="prefill-window"),
        # a long prompt of one request, chunk by chunk at page size 32: this chunk is far in
        dict(_prefill(1, 512, l8b, 32, start=8192), name="chunk-one"),
        # continuation chunks of a batch at the 70B head shape
        dict(_prefill(4, 512, l70b, 64, start=4096), name="chunk-batch"),
        # latent layers, decode batch: projections, cache write and attention over the latent cache
        dict(_latent_decode(128, 16, 64, 512, 8192), name="latent-decode"),
        # latent layers, prompts of four requests
        dict(_latent_prefill(4, 2048, 16, 64), name="latent-prefill"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(["decode", "decode", "prefill", "chunk", "latent-decode", "latent-prefill"])
        block = rng.choice([32, 64])
        if kind == "decode":
            lo = _log(rng, 64, 4096)
            window = rng.choice([0, 0, 0, 512, 1024, 4096])
            graph = rng.random() < 0.6
            users = _log(rng, 1, 160)
            heads = rng.choice(_HEADS)
            bfp8 = rng.random() < 0.3 and heads[2] != 256
            case = _decode(users, heads, block, lo, min(32768, _log(rng, lo, 32 * lo)), layers=4 if graph else 1,
                           graph=graph, bfp8=bfp8, window=window, sinks=window > 0 and rng.random() < 0.5,
                           parked=rng.choice([0, 0, users // 6]))
        elif kind == "prefill":
            case = _prefill(_log(rng, 1, 8), 32 * _log(rng, 1, 256), rng.choice(_HEADS), block,
                            window=rng.choice([0, 0, 512, 1024]))
        elif kind == "chunk":
            case = _prefill(_log(rng, 1, 8), 32 * _log(rng, 1, 64), rng.choice(_HEADS), block,
                            start=64 * _log(rng, 4, 256), bfp8=rng.random() < 0.4)
            if case["bfp8"] and case["head_size"] == 256:
                continue
        elif kind == "latent-decode":
            lo = _log(rng, 128, 4096)
            case = _latent_decode(_log(rng, 1, 160), rng.choice([16, 16, 32, 128]), block, lo, min(32768, _log(rng, lo, 16 * lo)))
        else:
            case = _latent_prefill(_log(rng, 1, 4), 32 * _log(rng, 1, 128), rng.choice([16, 16, 32]), block)
        w = work(case)
        if w["bytes"] <= _MAX_BYTES and w["flops"] <= _MAX_FLOPS:
            return case


# --------------------------------------------------------------------------- #
# sizes
# --------------------------------------------------------------------------- #
def _contexts(case):
    """Tokens in the cache before the step, one entry per active user."""
    n = case["users"] - case.get("parked", 0)
    lo, hi = case["ctx_lo"], case["ctx_hi"]
    return [int(round(lo * (hi / lo) ** ((i + 0.5) / n))) for i in range(n)]


def work(case):
    kind = case["kind"]
    hq = case["q_heads"]
    if kind == "decode":
        hkv, d = case["kv_heads"], case["head_size"]
        seen = [min(c + 1, case["window"] or c + 1) for c in _contexts(case)]
        per = 17 / 16 if case["bfp8"] else 2
        users = len(seen)
        # attended K / V once, the new token's K / V read and written, query, output, table entries
        nbytes = sum(seen) * hkv * d * 2 * per + users * hkv * d * 2 * (2 + per) + users * hq * d * 4 \
            + sum(-(-s // case["block"]) for s in seen) * 4
        return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * 4.0 * d * hq * sum(seen)}
    if kind == "prefill":
        b, s, hkv, d, start, window = (case[k] for k in ("users", "tokens", "kv_heads", "head_size", "start", "window"))
        per = 17 / 16 if case["bfp8"] else 2
        pairs = s * start + s * (s + 1) // 2
        if window and window < s:
            pairs = window * (window + 1) // 2 + (s - window) * window
        nbytes = b * (s * hq * d * 4 + s * hkv * d * 2 * (2 + per) + start * hkv * d * 2 * per)
        return {"bytes": nbytes, "flops": 4.0 * d * hq * b * pairs}
    lat, rope, nope, vh = _LATENT, _ROPE, _NOPE, _VHEAD
    weights = hq * lat * (nope + vh) * 2
    if kind == "latent-decode":
        seen = [c + 1 for c in _contexts(case)]
        rows, keys, pairs = len(seen), sum(seen), sum(seen)
    else:
        rows = case["users"] * case["tokens"]
        keys, pairs = rows, case["users"] * case["tokens"] * (case["tokens"] + 1) // 2
    per_row = hq * (nope + rope + vh) * 2 + 2 * (lat + rope) * 2
    kv_read = keys * (lat + rope) * 2 if kind == "latent-decode" else 0
    return {"bytes": weights + rows * per_row + kv_read,
            "flops": 2.0 * hq * (pairs * (2 * lat + rope) + rows * lat * (nope + vh))}


def tolerance(case):
    """Outputs are bfloat16 values of sums over probabilities rounded to bfloat16.  Measured against the
    same pass in 64 bits, for the listed and for drawn cases: 1.5e-3 .. 2.4e-3 (largest difference
    0.005 .. 0.05), and 2.9e-3 .. 4.4e-3 (0.006 .. 0.034) for the latent layers, whose absorbed query and
    latent output are rounded on the way as well.  Stated: four times that.  The caches are copies, or
    quantised copies in whole numbers: they do not differ."""
    if case["kind"].startswith("latent"):
        return {"rel": 1.6e-2, "max": 0.15}
    return {"rel": 1e-2, "max": 0.15}


# --------------------------------------------------------------------------- #
# inputs
# --------------------------------------------------------------------------- #
def _randn(gen, *shape, gain=1.0):
    return (torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * gain).to(torch.bfloat16)


def _pool(host, need, block_width):
    """Block tables for users that hold ``need`` blocks each, out of one shuffled pool with block 0 as
    the null block; (blocks in the pool, [users, block_width] int32)."""
    total = sum(need)
    blocks = total + max(8, total // 8) + 1
    order = host.permutation(blocks - 1)[:total] + 1
    table = np.zeros((len(need), block_width), dtype=np.int32)
    at = 0
    for u, n in enumerate(need):
        table[u, :n] = order[at : at + n]
        at += n
    return blocks, table


def _caches(gen, case, layers, blocks):
    """K and V caches of the layers, filled; [layers, blocks, kv_heads, rows, head_size] each."""
    from tt_xla_amd import TTAttentionBackend, custom_ops

    hkv, bs, d = case["kv_heads"], case["block"], case["head_size"]
    shape = TTAttentionBackend.get_kv_cache_storage_shape(blocks, bs, hkv, d, "bfp_bf8" if case["bfp8"] else "auto")
    pair = []
    for _ in range(2):
        cache = torch.empty((layers,) + tuple(shape), dtype=torch.uint8 if case["bfp8"] else torch.bfloat16, device="cuda")
        gain = torch.ones(hkv, 1, d, device="cuda", dtype=torch.bfloat16)
        if case["bfp8"]:  # one channel in a hundred is an outlier of the size that the option meets
            gain.view(-1)[torch.randperm(hkv * d, generator=gen, device="cuda")[: max(1, hkv * d // 100)]] = 20
        for n in range(layers):
            filled = torch.randn(blocks, hkv, bs, d, generator=gen, device="cuda", dtype=torch.bfloat16) * gain
            cache[n].copy_(custom_ops.bfp8_pack_cache(filled) if case["bfp8"] else filled)
        pair.append(cache)
    return pair


def _impl(case, sinks=None):
    from tt_xla_amd import TTAttentionBackendImpl

    return TTAttentionBackendImpl(case["q_heads"], case["head_size"], case["head_size"] ** -0.5, case["kv_heads"],
                                  None, case["window"] or None, "auto", sinks=sinks)


def _prepare_decode(case, gen, host):
    from tt_xla_amd.metadata import PagedMetadataBuilder

    users, layers, bs = case["users"], case["layers"], case["block"]
    hq, hkv, d = case["q_heads"], case["kv_heads"], case["head_size"]
    ctx = host.permutation(np.array(_contexts(case), dtype=np.int64))
    width = -(-(case["ctx_hi"] + 1) // bs)
    blocks, table = _pool(host, [int(c) // bs + 1 for c in ctx], width)
    builder = PagedMetadataBuilder(bs, width, min(2048, width * bs), device="cuda")
    meta = builder.prepare(table, ctx, np.ones(len(ctx), dtype=np.int64), target_num_reqs=users).metadata
    k_cache, v_cache = _caches(gen, case, layers, blocks)
    q, k, v = _randn(gen, layers, users, hq * d), _randn(gen, layers, users, hkv * d), _randn(gen, layers, users, hkv * d)
    out = torch.empty(layers, users, hq * d, dtype=torch.bfloat16, device="cuda")
    impls = [_impl(case, torch.randn(hq, generator=gen, device="cuda") if case["sinks"] else None) for _ in range(layers)]
    views = [(impls[n], q[n], k[n], v[n], [k_cache[n], v_cache[n]], out[n]) for n in range(layers)]

    def step():
        for impl, qn, kn, vn, kv, on in views:
            impl.forward(None, qn, kn, vn, kv, meta, output=on)

    state = {"step": step, "outputs": (out, k_cache, v_cache), "keep": (builder, meta)}
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            step()
        state["step"] = graph.replay
        state["keep"] += (graph, views)
    return state


def _prepare_prefill(case, gen, host):
    from tt_xla_amd.metadata import PagedMetadataBuilder

    users, s, bs, start = case["users"], case["tokens"], case["block"], case["start"]
    hq, hkv, d = case["q_heads"], case["kv_heads"], case["head_size"]
    width = -(-(start + s) // bs)
    blocks, table = _pool(host, [width] * users, width)
    # the step budget is the pass; the read table has room for the tokens to come
    builder = PagedMetadataBuilder(bs, width + -(-s // bs), 1 << (s - 1).bit_length(), device="cuda")
    meta = builder.prepare(table, np.full(users, start), np.full(users, s)).metadata
    k_cache, v_cache = _caches(gen, case, 1, blocks)
    q, k, v = _randn(gen, users * s, hq * d), _randn(gen, users * s, hkv * d), _randn(gen, users * s, hkv * d)
    out = torch.empty(users * s, hq * d, dtype=torch.bfloat16, device="cuda")
    impl, kv = _impl(case), [k_cache[0], v_cache[0]]

    def step():
        impl.forward(None, q, k, v, kv, meta, output=out)

    return {"step": step, "outputs": (out, k_cache, v_cache), "keep": (builder, meta)}


def _prepare_latent(case, gen, host):
    from tt_xla_amd import TTMetadata
    from tt_xla_amd.attention_mla import TTMLAAttentionBackend, TTMLAAttentionBackendImpl

    users, n, bs = case["users"], case["q_heads"], case["block"]
    decode = case["kind"] == "latent-decode"
    s = 1 if decode else case["tokens"]
    pos = host.permutation(np.array(_contexts(case))) if decode else np.full(users, s - 1)
    width = -(-(int(pos.max()) + 1) // bs)
    blocks, table = _pool(host, [int(p) // bs + 1 for p in pos], width)
    layer = types.SimpleNamespace(W_UK_T=_randn(gen, n, _NOPE, _LATENT, gain=_NOPE**-0.5),
                                  W_UV=_randn(gen, n, _LATENT, _VHEAD, gain=_LATENT**-0.5))
    impl = TTMLAAttentionBackendImpl(
        num_heads=n, head_size=_LATENT + _ROPE, scale=(_NOPE + _ROPE) ** -0.5, num_kv_heads=1, alibi_slopes=None,
        sliding_window=None, kv_cache_dtype="auto", logits_soft_cap=None, attn_type="decoder",
        kv_sharing_target_layer_name=None, kv_lora_rank=_LATENT, qk_nope_head_dim=_NOPE, qk_rope_head_dim=_ROPE,
        qk_head_dim=_NOPE + _ROPE, v_head_dim=_VHEAD)
    shape = TTMLAAttentionBackend.get_kv_cache_shape(blocks, bs, 1, _LATENT + _ROPE)
    cache = torch.randn(shape, generator=gen, device="cuda", dtype=torch.bfloat16)
    table = torch.from_numpy(table).cuda()
    meta = TTMetadata(cache_position=torch.from_numpy(pos.astype(np.int32)).cuda(), page_table=table,
                      fill_page_table=table, is_causal=True)
    q = (_randn(gen, users * s, n, _NOPE), _randn(gen, users * s, n, _ROPE))
    kv_c, k_pe = _randn(gen, users * s, _LATENT), _randn(gen, users * s, 1, _ROPE)
    out = torch.empty(users * s, n * _VHEAD, dtype=torch.bfloat16, device="cuda")

    def step():
        impl.forward(q, kv_c, k_pe, cache, meta, layer, output=out)

    return {"step": step, "outputs": (out, cache), "keep": (layer, meta)}


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    host = np.random.default_rng(seed)
    kind = case["kind"]
    make = _prepare_decode if kind == "decode" else _prepare_prefill if kind == "prefill" else _prepare_latent
    return make(case, gen, host)


def run(state):
    state["step"]()
    return state["outputs"]
