"""The calls that a user of this framework makes, as cases that can be timed and compared.

Each case names an operation (``op``) and its sizes.  ``prepare`` makes what a program holds
before the call (inputs, cache, model, captured graph), ``run`` makes one call through the public
entry points, ``exact`` computes the same outputs in 64 bits with plain torch.

Operations and what they stand for:

* ``prefill``: one layer's one-shot prefill of a whole prompt (compressor + attention).
* ``stream``: one layer's chunked prefill of a prompt into an empty two-pool cache.
* ``decode_graph``: one layer's decode steps on device counters, replayed from a HIP graph.
* ``decode_eager``: one decode step through the swapped layer's attention core.
* ``active``: new rows over the full keys and values of a plain (uncompressed) cache, whose
  summaries are made anew in every call.
* ``streams``: the stream-level interface: sliding window, dense or routed summaries, merge.
* ``decoder_step``: a decode step of the 4-bit decoder (a few of its layers, the lm_head),
  replayed from a HIP graph with device counters.
* ``decoder_prefill``: a prompt through the same decoder, to the logits of its last position.

Windows: 64 tokens is the benchmark configurations' window, 128 the default of
``QwenButterflyConfig`` and ``CompressedKVCache``.
"""
import math

import torch
import torch.nn.functional as F

import butterfly_amd as bf
from butterfly_amd import decoder as dec

_DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


# --------------------------------------------------------------------------- cases
def listed():
    return [
        # the reference check's layer: fp32, 4096 tokens, layer 3 of its five stages
        dict(name="prefill_fp32_4k", op="prefill", dtype="fp32", batch=1, tokens=4096, hq=8, hkv=2, d=128, window=64,
             block=128, layer=3, rule="causal_shift"),
        # the headline layer: a 64k-token prompt in bf16
        dict(name="prefill_64k", op="prefill", dtype="bf16", batch=1, tokens=65536, hq=8, hkv=2, d=128, window=64,
             block=128, layer=3, rule="causal_shift"),
        # the integration's default settings (128-token window, xor partners), two ragged prompts
        dict(name="prefill_window128", op="prefill", dtype="bf16", batch=2, tokens=10007, hq=16, hkv=4, d=128,
             window=128, block=128, layer=5, rule="xor"),
        # long-context ingestion: 384-token chunks into a ring that holds several of them
        dict(name="stream_384", op="stream", batch=1, tokens=23040, chunk=384, max_chunk=4096, hq=16, hkv=4, d=256,
             window=64, cache_window=64, block=128, layer=5, rule="causal_shift"),
        # chunked prefill with the default cache and config (128-token windows, 512-token chunks), ragged end
        dict(name="stream_window128", op="stream", batch=1, tokens=20011, chunk=512, max_chunk=512, hq=16, hkv=4,
             d=256, window=128, cache_window=128, block=128, layer=5, rule="xor"),
        # batched decode at a 128k context, 64 steps in one graph
        dict(name="decode_graph_b32", op="decode_graph", batch=32, context=131072, steps=64, hq=8, hkv=2, d=128,
             window=64, block=128, layer=3, rule="causal_shift"),
        # the smallest call: one token through a layer with the default settings
        dict(name="decode_window128", op="decode_eager", batch=1, context=5000, hq=16, hkv=4, d=128, window=128,
             cache_window=128, block=128, layer=5, rule="xor"),
        # a chunk of a prompt over a plain cache of 32k tokens, default window
        dict(name="active_512_of_32k", op="active", dtype="bf16", batch=1, tokens=32768, rows=512, hq=16, hkv=4, d=128,
             window=128, block=128, layer=5, rule="xor"),
        # the stream-level ablation: window stream + every earlier summary + merge
        dict(name="streams_dense_8k", op="streams", batch=1, tokens=8192, hq=8, hkv=2, d=128, window=64, block=128,
             layer=3, rule="causal_shift", routed=False),
        # one sequence's decode step of the 4-bit decoder
        dict(name="decoder_step_b1", op="decoder_step", batch=1, context=4096, layers=4),
        # a small serving batch's decode step
        dict(name="decoder_step_b8", op="decoder_step", batch=8, context=1000, layers=4),
        # a prompt through the decoder
        dict(name="decoder_prefill_8k", op="decoder_prefill", batch=1, tokens=8192, layers=4),
    ]


def _log(rng, lo, hi):
    """An integer between lo and hi, spread evenly over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["prefill", "prefill", "stream", "decode_graph", "decode_eager", "active", "streams",
                     "decoder_step", "decoder_prefill"])
    rule = rng.choice(["causal_shift", "xor"])
    layer = rng.randrange(24)
    hkv = rng.choice([1, 2, 4])
    d = rng.choice([64, 128, 256])
    common = dict(hkv=hkv, hq=hkv * rng.choice([1, 2, 4, 8]), d=d, window=rng.choice([64, 128, rng.randint(16, 128)]),
                  block=rng.choice([64, 128, 128, 256]), layer=layer, rule=rule)
    if op in ("prefill", "active"):
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
        c = dict(common, op=op, dtype=dtype, batch=rng.choice([1, 1, 2, 4]))
        if dtype == "fp32":   # the check's head shapes
            c["d"], c["hq"] = min(d, 128), min(c["hq"], 4 * hkv)
        # no more work than the headline layer's (fp32: an eighth of it)
        per = c["batch"] * (c["hq"] + hkv) * c["d"]
        most = 65536 * 10 * 128 // (per * (8 if dtype == "fp32" else 1))
        c["tokens"] = _log(rng, 64, max(64, min(65536, most)))
        if op == "active":
            c["rows"] = _log(rng, 1, min(512, c["tokens"]))
        return c
    if op == "stream":
        w = common["window"]
        chunk = _log(rng, 64, 1024)
        return dict(common, op="stream", batch=1, chunk=chunk, max_chunk=max(chunk, rng.choice([512, 4096])),
                    cache_window=max(w, rng.choice([64, 128])), tokens=chunk * rng.randint(2, 47) + rng.randrange(chunk))
    if op == "decode_graph":
        return dict(common, op="decode_graph", batch=_log(rng, 1, 32), context=_log(rng, 1000, 131072),
                    steps=rng.randint(16, 64), window=min(64, common["window"]))
    if op == "decode_eager":
        return dict(common, op="decode_eager", batch=_log(rng, 1, 32), context=_log(rng, 300, 16384), cache_window=128)
    if op == "streams":
        return dict(common, op="streams", batch=rng.choice([1, 2]), tokens=_log(rng, 128, 8192), d=min(d, 128),
                    hq=min(common["hq"], 4 * hkv, 8), routed=rng.random() < 0.5)
    if op == "decoder_step":
        return dict(op="decoder_step", batch=_log(rng, 1, 16), context=_log(rng, 100, 1000), layers=rng.randint(2, 4))
    return dict(op="decoder_prefill", batch=rng.choice([1, 1, 2]), tokens=_log(rng, 16, 4096), layers=rng.randint(2, 4))


# --------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=g, device="cuda").to(dtype)


def _qkv(c, seed, dtype, rows=None):
    """q, k ~ N(0, 1) (k with per-channel scales from U(0.5, 2): outlier channels), v ~ N(0, 1)."""
    g = _gen(seed)
    t, b = c["tokens"], c["batch"]
    q = _randn(g, b, c["hq"], rows or t, c["d"], dtype=dtype)
    ch = torch.rand(c["hkv"], 1, c["d"], generator=g, device="cuda") * 1.5 + 0.5
    k = (torch.randn(b, c["hkv"], t, c["d"], generator=g, device="cuda") * ch).to(dtype)
    return q, k, _randn(g, b, c["hkv"], t, c["d"], dtype=dtype)


def _config(c):
    return bf.compressed_butterfly_config(block_partner_rule=c["rule"], block_size=c["block"],
                                          compressed_local_window_tokens=c["window"])


def _layout(c, tokens):
    return bf.build_block_butterfly_layout(
        seq_len=tokens, block_size=c["block"], num_key_value_heads=c["hkv"], num_key_value_groups=c["hq"] // c["hkv"],
        layer_idx=c["layer"], local_window_blocks=1, sink_count=1, partner_count=1, partner_rule=c["rule"])


def _restored(c):
    """Counters of a cache after ``context`` tokens: (summaries, tail tokens kept)."""
    w = c.get("cache_window", c["window"])
    count = max(0, (c["context"] - w) // c["block"])
    return count, c["context"] - max(0, count - 1) * c["block"]


def _decode_inputs(c, seed):
    count, tail = _restored(c)
    g, b, n = _gen(seed), c["batch"], c.get("steps", 1)
    kv = [_randn(g, b, c["hkv"], m, c["d"]) for m in (tail, tail, count, count)]
    return kv, _randn(g, n, b, c["hq"], 1, c["d"]), _randn(g, n, b, c["hkv"], 1, c["d"]), \
        _randn(g, n, b, c["hkv"], 1, c["d"])


def _restored_cache(c, kv):
    # room in the pool for a long run of further steps
    cache = bf.CompressedKVCache(block_size=c["block"], local_window_tokens=c.get("cache_window", c["window"]),
                                 max_kv_size=c["context"] + (1 << 20), max_chunk_size=512)
    cache.state = tuple(kv)
    cache.meta_state = (str(c["block"]), str(cache.local_window_tokens), str(c["context"]),
                        str(kv[2].shape[2] * c["block"]))
    return cache, cache.ring_state()


def _model(c, seed):
    cfg = dec.DecoderConfig(num_layers=c["layers"])
    model = dec.Decoder(cfg, seed=seed, device="cuda")
    bf.swap_qwen_attention_with_butterfly(model, cfg=bf.compressed_butterfly_config())
    tokens = torch.randint(0, cfg.vocab_size, (c["batch"], c.get("tokens", c.get("context"))), generator=_gen(seed + 1),
                           device="cuda")
    return model, tokens


def _model_caches(model, tokens, extra):
    caches = [None] * len(model.layers)
    bf.install_compressed_kv_caches(model, caches, block_size=128, local_window_tokens=64, max_kv_size=tokens + extra,
                                    max_chunk_size=max(512, tokens))
    return caches


_STEP_ROOM = 65536   # positions that a decoder_step state can advance through


def prepare(case, seed):
    c = case
    op = c["op"]
    if op == "prefill":
        q, k, v = _qkv(c, seed, _DTYPES[c["dtype"]])
        return dict(c=c, q=q, k=k, v=v, layout=_layout(c, c["tokens"]))
    if op == "active":
        q, k, v = _qkv(c, seed, _DTYPES[c["dtype"]], rows=c["rows"])
        return dict(c=c, q=q, k=k, v=v, core=bf.ButterflyAttentionCore(_config(c), c["layer"]))
    if op == "stream":
        chunks = bf.split_chunks(*_qkv(c, seed, torch.bfloat16), c["chunk"])
        return dict(c=c, chunks=chunks, core=bf.ButterflyAttentionCore(_config(c), c["layer"]))
    if op == "streams":
        q, k, v = _qkv(c, seed, torch.bfloat16)
        routed = None
        if c["routed"]:
            n = -(-c["tokens"] // c["block"])
            row = torch.tensor([_routed_row(b, n, c["layer"], c["rule"]) for b in range(n)], dtype=torch.int32)
            routed = row.unsqueeze(0).expand(c["hq"], -1, -1).contiguous().cuda()
        return dict(c=c, q=q, k=k, v=v, routed=routed)
    if op == "decode_eager":
        kv, q, k, v = _decode_inputs(c, seed)
        cache, st = _restored_cache(c, kv)
        return dict(c=c, q=q[0], k=k[0], v=v[0], cache=cache, st=st,
                    core=bf.ButterflyAttentionCore(_config(c), c["layer"]))
    if op == "decode_graph":
        kv, q, k, v = _decode_inputs(c, seed)
        cache, st = _restored_cache(c, kv)
        cache.use_device_counters()
        out = torch.empty_like(q)

        def steps():
            for i in range(c["steps"]):
                cache.decode_step(q[i], k[i], v[i], layer_idx=c["layer"], local_window_tokens=c["window"],
                                  partner_rule=c["rule"], out=out[i])

        return dict(c=c, q=q, k=k, v=v, cache=cache, st=st, out=out, graph=_captured(steps))
    model, tokens = _model(c, seed)
    if op == "decoder_prefill":
        return dict(c=c, model=model, tokens=tokens)
    # decoder_step: the prompt, one eager step, then the step as a graph (input token fixed, position advancing)
    ctx = c["context"]
    caches = _model_caches(model, ctx, _STEP_ROOM)
    model.forward(tokens, caches, 0)
    for cache in caches:
        cache.use_device_counters()
    tok = tokens[:, :1].clone()
    pos = torch.tensor([ctx], dtype=torch.long, device="cuda")
    cos, sin = dec.rope_cos_sin(torch.arange(ctx + _STEP_ROOM, device="cuda"), model.cfg.head_dim, model.cfg.rope_theta)
    rope = dec.RopeTable(cos, sin, pos)
    got = {}

    @torch.no_grad()
    def step():
        x, m = F.embedding(tok, model.embed_tokens), None
        for layer, cache in zip(model.layers, caches):
            x, m = layer.forward_split(x, m, pos, cache, rope)
        xl, ml, norm = x[:, -1], m[:, -1], model.norm
        if dec.norm_q4_fits(xl, model.lm_head):
            got["logits"] = dec.add_rms_norm_q4_gemv(xl, ml, norm.weight, norm.eps, model.lm_head)[1]
        else:
            got["logits"] = model.lm_head(dec.add_rms_norm(xl, ml, norm.weight, norm.eps)[1])
        pos.add_(1)

    step()
    return dict(c=c, model=model, caches=caches, tok=tok, rope=rope, graph=_captured(step), logits=got["logits"])


def _captured(fn):
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            fn()
    torch.cuda.current_stream().wait_stream(side)
    return graph


# --------------------------------------------------------------------------- one call
def run(state):
    c = state["c"]
    op = c["op"]
    if op == "prefill":
        return bf.compressed_butterfly_attention(state["q"], state["k"], state["v"], layout=state["layout"],
                                                 local_window_tokens=c["window"])[0]
    if op == "active":
        return state["core"].attend_full(state["q"], state["k"], state["v"])
    if op == "stream":
        # a new prompt: an empty cache, filled chunk by chunk
        cache = bf.CompressedKVCache(block_size=c["block"], local_window_tokens=c["cache_window"],
                                     max_kv_size=c["tokens"], max_chunk_size=c["max_chunk"])
        outs = bf.chunked_prefill(state["core"], state["chunks"], cache)
        st = cache.ring_state()
        return {"out": outs, "tail": [st.ring_k, st.ring_v], "pool": [st.pool_k, st.pool_v]}
    if op == "streams":
        q, k, v, n = state["q"], state["k"], state["v"], -(-c["tokens"] // c["block"])
        scale = c["d"] ** -0.5
        ks, vs = bf.block_mean_summaries(k, seq_len=c["tokens"], block_size=c["block"], num_blocks=n, x2=v)
        near = bf.swa_stream_attention(q, k, v, n_win=c["window"], scale=scale)
        far = bf.compressed_stream_attention(q, ks, vs, block_size=c["block"], scale=scale,
                                             routed_indices=state["routed"])
        return {"out": bf.online_softmax_merge(near, far), "near": near[0], "far": far[0], "near_l": near[1]}
    if op == "decode_eager":
        out = state["core"](state["q"], state["k"], state["v"], state["cache"])
        st = state["st"]
        return {"out": out, "tail": [st.ring_k, st.ring_v], "pool": [st.pool_k, st.pool_v]}
    if op == "decode_graph":
        state["graph"].replay()
        st = state["st"]
        return {"out": state["out"], "tail": [st.ring_k, st.ring_v], "pool": [st.pool_k, st.pool_v]}
    if op == "decoder_step":
        state["graph"].replay()
        return state["logits"]
    caches = _model_caches(state["model"], c["tokens"], 512)
    return state["model"].forward(state["tokens"], caches, 0)


# --------------------------------------------------------------------------- what a call cannot do without
def _keys(c, t):
    """Window keys that t prompt queries attend to."""
    w = min(c["window"], t)
    return w * (w + 1) // 2 + (t - w) * w


def _weights(layers):
    cfg = dec.DecoderConfig()
    h, f = cfg.hidden_size, cfg.intermediate_size
    return layers * (h * (cfg.num_heads + 2 * cfg.num_kv_heads) * cfg.head_dim + cfg.num_heads * cfg.head_dim * h
                     + 3 * h * f), cfg.vocab_size * h


def work(case):
    c = case
    op = c["op"]
    if op in ("prefill", "stream", "streams"):
        e = 4 if c.get("dtype") == "fp32" else 2
        b, t, d, hq, hkv = c["batch"], c["tokens"], c["d"], c["hq"], c["hkv"]
        n = -(-t // c["block"])
        rows = 2 * b * t * (hq + hkv) * d * e
        if op == "streams":
            far = 2 * t if c["routed"] else sum(i // c["block"] for i in range(t))
            # the two streams' outputs and the merged one in fp32
            return {"bytes": rows + b * t * hq * d * (2 + 4), "flops": 4 * d * b * hq * (_keys(c, t) + far)}
        return {"bytes": rows + 2 * b * n * hkv * d * e, "flops": 4 * d * b * hq * (_keys(c, t) + 2 * t)}
    if op == "active":
        e = 4 if c["dtype"] == "fp32" else 2
        return {"bytes": e * c["batch"] * c["d"] * (2 * c["rows"] * c["hq"] + 2 * c["tokens"] * c["hkv"]),
                "flops": 4 * c["d"] * c["batch"] * c["hq"] * c["rows"] * (c["window"] + 2)}
    if op in ("decode_eager", "decode_graph"):
        n = c.get("steps", 1) * c["batch"]
        return {"bytes": 2 * n * c["d"] * (2 * c["hq"] + c["hkv"] * (2 * c["window"] + 4 + 4)),
                "flops": 4 * n * c["d"] * c["hq"] * (c["window"] + 2)}
    layers, head = _weights(c["layers"])
    code = 0.5 + 4 / 64   # bytes of a 4-bit weight with its share of the group's scale and bias
    rows = c["batch"] * (c["tokens"] if op == "decoder_prefill" else 1)
    return {"bytes": (layers + head) * code + rows * 2048 * 2 + c["batch"] * 151936 * 2,
            "flops": 2 * rows * layers + 2 * c["batch"] * head}


def tolerance(case):
    op = case["op"]
    if op in ("decoder_step", "decoder_prefill"):
        return {"rel": 0.03, "max": 0.3}      # a bf16 rounding in one layer travels through the others
    if case.get("dtype") == "fp32":
        return {"rel": 4e-6, "max": 1e-4}
    return {"rel": 1e-2, "max": 0.2}


# --------------------------------------------------------------------------- the same in 64 bits
def _stages(n):
    return 1 if n <= 1 else int(math.ceil(math.log2(n)))


def _routed_row(b, n, layer, rule):
    """Blocks before b on its routed row (previous, partner, first; each once), -1 padded."""
    bit = layer % _stages(n)
    partner = b - (1 << bit) if rule == "causal_shift" else b ^ (1 << bit)
    row = []
    for x in (b - 1, partner, 0):
        if 0 <= x < b and x < n and x not in row:
            row.append(x)
    return row + [-1] * (3 - len(row))


def _means64(x, block, dtype=None):
    """Block means [B, H, N, d] in 64 bits, rounded to the cache's type where that is given."""
    t = x.shape[2]
    full = t // block * block
    m = x[:, :, :full].double().unflatten(2, (full // block, block)).mean(3) if full else \
        x.new_zeros((*x.shape[:2], 0, x.shape[3]), dtype=torch.float64)
    if full < t:
        m = torch.cat([m, x[:, :, full:].double().mean(2, keepdim=True)], 2)
    return m if dtype is None else m.to(dtype).double()


def _rows64(q, k, v, ks, vs, c, *, pos0, kv_len, nsum, token_cutoff, key0=0, window=True, far=True, dense=False):
    """Attention of the queries at [pos0, pos0 + q_len) in 64 bits; k/v hold positions from key0 on.

    Returns (normalised output, row sums, row maxima)."""
    b, hq, tq, d = q.shape
    hkv, w, bs = k.shape[1], c["window"], c["block"]
    g, n, dev = hq // hkv, -(-kv_len // bs), q.device
    table = None
    if far and not dense:
        table = torch.tensor([_routed_row(i, n, c["layer"], c["rule"]) for i in range(n)], device=dev)
    outs, sums, tops = [], [], []
    step = max(64, 4096 // max(1, b * hkv * d // 1024) // 64 * 64)
    for s in range(0, tq, step):
        m = min(step, tq - s)
        pad = -m % 64
        p = torch.arange(pos0 + s, pos0 + s + m + pad, device=dev)
        qq = F.pad(q[:, :, s:s + m].double(), (0, 0, 0, pad)).view(b, hkv, g, -1, 64, d) * d ** -0.5
        groups = qq.shape[3]
        scores, values = [], []
        if window:
            at = p.view(-1, 64)[:, :1] - w + 1 + torch.arange(w + 63, device=dev)          # [groups, w + 63]
            rows = (at - key0).clamp(0, k.shape[2] - 1)
            kk, vv = k[:, :, rows].double(), v[:, :, rows].double()                          # [b, hkv, groups, keys, d]
            sc = torch.matmul(qq.transpose(2, 3).reshape(b, hkv, groups, g * 64, d), kk.transpose(3, 4).contiguous())
            sc = sc.view(b, hkv, groups, g, 64, -1)
            pq = p.view(-1, 64)
            ok = (at[:, None] <= pq[:, :, None]) & (at[:, None] > pq[:, :, None] - w) & (at[:, None] >= 0)
            scores.append(sc.masked_fill(~ok[None, None, :, None], -math.inf))
            values.append(vv)
        if far and dense:
            kk, vv = ks[:, :, None].expand(-1, -1, groups, -1, -1), vs[:, :, None].expand(-1, -1, groups, -1, -1)
            sc = torch.matmul(qq.transpose(2, 3).reshape(b, hkv, groups, g * 64, d), kk.transpose(3, 4))
            ok = torch.arange(ks.shape[2], device=dev) < (p // bs).view(-1, 64, 1)
            scores.append(sc.view(b, hkv, groups, g, 64, -1).masked_fill(~ok[None, None, :, None], -math.inf))
            values.append(vv)
        if far and not dense:
            blk = (p // bs).clamp(max=n - 1)
            cand = table[blk]                                                                # [m, 3]
            cut = (p if token_cutoff == "token" else blk * bs) - w + 1
            ok = (cand >= 0) & (cand < nsum)
            if token_cutoff != "none":
                ok = ok & ((cand + 1) * bs <= cut[:, None])
            kk, vv = ks[:, :, cand.clamp(0, ks.shape[2] - 1)], vs[:, :, cand.clamp(0, vs.shape[2] - 1)]
            kk, vv = (x.view(b, hkv, groups, 64, 3, d) for x in (kk, vv))
            sc = (qq.unsqueeze(-2) * kk[:, :, None]).sum(-1).transpose(2, 3)                 # [b, hkv, groups, g, 64, 3]
            scores.append(sc.masked_fill(~ok.view(groups, 64, 3)[None, None, :, None], -math.inf))
            values.append(vv)
        sc = torch.cat(scores, -1)
        top = sc.amax(-1, keepdim=True)
        top = torch.where(top == -math.inf, torch.zeros_like(top), top)
        e = torch.exp(sc - top)
        l, o, at0 = e.sum(-1, keepdim=True), 0.0, 0
        for x, vv in zip(scores, values):
            part = e[..., at0:at0 + x.shape[-1]]
            at0 += x.shape[-1]
            if vv.dim() == 6:
                o = o + (part.unsqueeze(-1) * vv[:, :, :, None]).sum(-2)
            else:
                o = o + torch.matmul(part.reshape(b, hkv, groups, g * 64, -1), vv).view(b, hkv, groups, g, 64, d)
        o = o / l.clamp_min(1e-300)
        put = lambda x: x.transpose(2, 3).reshape(b, hq, m + pad, -1)[:, :, :m]  # noqa: E731
        outs.append(put(o)), sums.append(put(l)), tops.append(put(top))
    return torch.cat(outs, 2), torch.cat(sums, 2), torch.cat(tops, 2)


def _decode64(c, kv, q, k, v):
    """The steps of a restored cache in 64 bits: [steps, B, Hq, 1, d]."""
    count, _ = _restored(c)
    ctx, bs, cw = c["context"], c["block"], c.get("cache_window", c["window"])
    key0 = ctx - kv[0].shape[2]
    kk = torch.cat([kv[0], k.permute(1, 2, 0, 3, 4).flatten(2, 3)], 2)
    vv = torch.cat([kv[1], v.permute(1, 2, 0, 3, 4).flatten(2, 3)], 2)
    ks, vs = kv[2].double(), kv[3].double()
    outs = []
    for i in range(q.shape[0]):
        offset = ctx + i + 1
        while (count + 1) * bs + cw <= offset:      # the blocks that left the cache's window
            lo = count * bs - key0
            ks, vs = (torch.cat([s, x[:, :, lo:lo + bs].double().mean(2, keepdim=True).to(x.dtype).double()], 2)
                      for s, x in ((ks, kk), (vs, vv)))
            count += 1
        outs.append(_rows64(q[i], kk, vv, ks, vs, c, pos0=offset - 1, kv_len=offset, nsum=count, key0=key0,
                            token_cutoff="token")[0])
    return torch.stack(outs)


class _Model64:
    """The decoder in 64 bits, from its 4-bit codes."""

    def __init__(self, model):
        self.cfg, self.model = model.cfg, model
        self.c = dict(window=64, block=128, rule="causal_shift")
        self.k, self.v = [None] * len(model.layers), [None] * len(model.layers)

    @staticmethod
    def lin(x, layer):
        codes = torch.stack([layer.packed & 0xF, layer.packed >> 4], -1).flatten(1).double()
        per = codes.view(codes.shape[0], -1, layer.group)
        w = per * layer.scale.double().unsqueeze(-1) + layer.bias.double().unsqueeze(-1)
        return x @ w.flatten(1).t()

    def norm(self, x, w):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + self.cfg.rms_eps) * w.double()

    def rope(self, x, pos):
        d = x.shape[-1]
        ang = pos.double()[:, None] / (self.cfg.rope_theta ** (torch.arange(0, d, 2, device=x.device).double() / d))
        cos, sin = torch.cat([ang, ang], -1).cos(), torch.cat([ang, ang], -1).sin()
        return x * cos + torch.cat([-x[..., d // 2:], x[..., :d // 2]], -1) * sin

    def forward(self, tokens, start):
        """Logits of the last position; appends to the keys and values of the calls before."""
        c, (b, t) = self.cfg, tokens.shape
        x = self.model.embed_tokens[tokens].double()
        pos = torch.arange(start, start + t, device=x.device)
        for i, layer in enumerate(self.model.layers):
            at, mlp = layer.self_attn.base, layer.mlp
            n = self.norm(x, layer.input_layernorm.weight)
            heads = lambda y, h: y.view(b, t, h, c.head_dim).transpose(1, 2)  # noqa: E731
            q = self.rope(self.norm(heads(self.lin(n, at.q_proj), c.num_heads), at.q_norm.weight), pos)
            k = self.rope(self.norm(heads(self.lin(n, at.k_proj), c.num_kv_heads), at.k_norm.weight), pos)
            v = heads(self.lin(n, at.v_proj), c.num_kv_heads)
            if start:
                k, v = torch.cat([self.k[i], k], 2), torch.cat([self.v[i], v], 2)
            self.k[i], self.v[i] = k, v
            kv_len = start + t
            nsum = max(0, (kv_len - 64) // 128) if start else -(-kv_len // 128)
            o = _rows64(q, k, v, _means64(k, 128), _means64(v, 128), dict(self.c, layer=i), pos0=start, kv_len=kv_len,
                        nsum=nsum, token_cutoff="token" if start else "block")[0]
            x = x + self.lin(o.transpose(1, 2).reshape(b, t, -1), at.o_proj)
            n = self.norm(x, layer.post_attention_layernorm.weight)
            x = x + self.lin(F.silu(self.lin(n, mlp.gate_proj)) * self.lin(n, mlp.up_proj), mlp.down_proj)
        return self.lin(self.norm(x[:, -1], self.model.norm.weight), self.model.lm_head)


@torch.no_grad()
def exact(case, seed):
    c = case
    op = c["op"]
    if op == "prefill":
        dt = _DTYPES[c["dtype"]]
        q, k, v = _qkv(c, seed, dt)
        n = -(-c["tokens"] // c["block"])
        return _rows64(q, k, v, _means64(k, c["block"], dt), _means64(v, c["block"], dt), c, pos0=0,
                       kv_len=c["tokens"], nsum=n, token_cutoff="block")[0]
    if op == "active":
        dt, t, r = _DTYPES[c["dtype"]], c["tokens"], c["rows"]
        q, k, v = _qkv(c, seed, dt, rows=r)
        n = -(-t // c["block"])
        return _rows64(q, k, v, _means64(k, c["block"], dt), _means64(v, c["block"], dt), c, pos0=t - r, kv_len=t,
                       nsum=n, token_cutoff="block" if r == t else "token")[0]
    if op == "stream":
        q, k, v = _qkv(c, seed, torch.bfloat16)
        t, ch, bs = c["tokens"], c["chunk"], c["block"]
        outs = []
        for s in range(0, t, ch):
            e = min(s + ch, t)
            if s == 0:   # the first chunk attends to its own tokens
                ks, vs = (_means64(x[:, :, :e], bs, x.dtype) for x in (k, v))
                args = dict(nsum=-(-e // bs), token_cutoff="block")
            else:
                count = max(0, (e - c["cache_window"]) // bs)
                ks, vs = (_means64(x[:, :, :max(1, count) * bs], bs, x.dtype) for x in (k, v))
                args = dict(nsum=count, token_cutoff="token")
            outs.append(_rows64(q[:, :, s:e], k[:, :, :e], v[:, :, :e], ks, vs, c, pos0=s, kv_len=e, **args)[0])
        return {"out": outs, "tail": [None, None], "pool": [None, None]}
    if op == "streams":
        q, k, v = _qkv(c, seed, torch.bfloat16)
        t, n = c["tokens"], -(-c["tokens"] // c["block"])
        ks, vs = (_means64(x, c["block"], x.dtype) for x in (k, v))
        args = dict(pos0=0, kv_len=t, nsum=n, token_cutoff="none", dense=not c["routed"])
        on, ln, mn = _rows64(q, k, v, ks, vs, c, far=False, **args)
        of, lf, mf = _rows64(q, k, v, ks, vs, c, window=False, **args)
        mf = torch.where(lf > 0, mf, torch.full_like(mf, -1e30))
        top = torch.maximum(mn, mf)
        wn, wf = ln * torch.exp(mn - top), lf * torch.exp(mf - top)
        return {"out": (wn * on + wf * of) / (wn + wf), "near": on, "far": of, "near_l": ln}
    if op in ("decode_eager", "decode_graph"):
        out = _decode64(c, *_decode_inputs(c, seed))
        return {"out": out[0] if op == "decode_eager" else out, "tail": [None, None], "pool": [None, None]}
    model, tokens = _model(c, seed)
    m = _Model64(model)
    if op == "decoder_prefill":
        return m.forward(tokens, 0)
    m.forward(tokens, 0)
    m.forward(tokens[:, :1], c["context"])           # the eager step
    return m.forward(tokens[:, :1], c["context"] + 1)
