"""GPU: the paged MFMA kernel (windows above 64, blocks below 64, the bf16 streams) against the oracle.

The oracle runs in float32 over the same bf16 inputs and the device's own bf16 summaries, so what
remains is the output's rounding to bf16 (half an ulp, at most 2^-8 of the value) and fp32
arithmetic: scores and weights carry a relative error of about 1e-6, times values of up to 5.
"""
from __future__ import annotations

import math

import pytest
import torch

import butterfly_amd as bf
from oracle import attention as oa, topology as tp

pytestmark = pytest.mark.gpu

BF16_ROUNDING = 2.0 ** -8
ABS = 5e-5


def _rand(seed, *shape):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).bfloat16()


def _layouts(t, bs, hkv, groups, layer, rule="causal_shift", **over):
    kw = dict(seq_len=t, block_size=bs, num_key_value_heads=hkv, num_key_value_groups=groups, layer_idx=layer,
              local_window_blocks=1, sink_count=1, partner_count=1, partner_rule=rule)
    kw.update(over)
    return bf.build_block_butterfly_layout(**kw), tp.build_layout(**kw)


def _check(got, want):
    got, want = got.float().cpu(), want.float()
    assert ((got - want).abs() <= BF16_ROUNDING * want.abs() + ABS).all(), (got - want).abs().max()


def _summaries(k, v, bs):
    t = k.shape[2]
    return [s.cpu().float() for s in bf.block_mean_summaries(k.cuda(), seq_len=t, block_size=bs,
                                                            num_blocks=-(-t // bs), x2=v.cuda())]


# b, hq, hkv, t, d, bs, W, layer, rule: page and tile edges of length and window, blocks that split a
# 64-position chunk or straddle two, every heads-per-workgroup form (from 256 units on: two and four
# heads) with groups that leave some of a workgroup's heads empty
CASES = [
    (1, 2, 1, 1, 128, 128, 128, 0, "xor"),
    (1, 4, 4, 65, 64, 128, 65, 1, "xor"),
    (1, 8, 2, 129, 128, 128, 128, 1, "causal_shift"),
    (2, 3, 1, 1000, 128, 128, 127, 2, "xor"),
    (1, 16, 2, 777, 64, 64, 200, 3, "benes"),
    (1, 8, 4, 1500, 256, 128, 128, 5, "xor"),
    (1, 2, 2, 700, 256, 256, 96, 2, "causal_shift"),
    (1, 4, 2, 2300, 128, 128, 1900, 1, "xor"),
    (1, 4, 1, 500, 128, 32, 33, 2, "causal_shift"),
    (1, 4, 2, 400, 64, 16, 64, 3, "xor"),
    (1, 4, 2, 450, 128, 48, 40, 3, "xor"),
    (1, 2, 1, 600, 64, 100, 130, 2, "causal_shift"),
    (2, 16, 4, 2113, 128, 128, 128, 5, "xor"),
    (3, 20, 4, 1501, 64, 128, 90, 4, "causal_shift"),
    (4, 8, 4, 1100, 128, 64, 128, 2, "xor"),
    (2, 12, 4, 2200, 256, 128, 128, 6, "causal_shift"),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x) for x in c))
def test_prefill(case):
    b, hq, hkv, t, d, bs, w, layer, rule = case
    q, k, v = _rand(t, b, hq, t, d), _rand(t + 1, b, hkv, t, d), _rand(t + 2, b, hkv, t, d)
    lay, ref = _layouts(t, bs, hkv, hq // hkv, layer, rule)
    ks, vs = _summaries(k, v, bs)
    want = oa.prefill(q.float(), k.float(), v.float(), layout=ref, W=w, k_summary=ks, v_summary=vs)
    _check(bf.compressed_butterfly_attention(q.cuda(), k.cuda(), v.cuda(), layout=lay, local_window_tokens=w)[0], want)


def test_wide_rows_and_scales():
    """A routed row of 13 slots, and scales that the W <= 64 kernel does not take."""
    b, hq, hkv, t, d, bs = 1, 4, 2, 1300, 64, 64
    q, k, v = _rand(1, b, hq, t, d), _rand(2, b, hkv, t, d), _rand(3, b, hkv, t, d)
    lay, ref = _layouts(t, bs, hkv, 2, 1, local_window_blocks=5, sink_count=3, partner_count=4)
    ks, vs = _summaries(k, v, bs)
    for scale, w in ((0.125, 64), (-0.1, 100), (0.0, 70)):
        want = oa.prefill(q.float() * (scale * d ** 0.5), k.float(), v.float(), layout=ref, W=w, k_summary=ks,
                          v_summary=vs)
        _check(bf.compressed_butterfly_attention(q.cuda(), k.cuda(), v.cuda(), layout=lay, local_window_tokens=w,
                                                 scale=scale)[0], want)


@pytest.mark.parametrize("d,w,bs,step,hq,hkv", [(128, 128, 128, 100, 8, 2), (64, 100, 64, 37, 4, 4),
                                                (256, 128, 128, 512, 16, 4), (128, 40, 32, 3, 4, 2)])
def test_ring_chunks(d, w, bs, step, hq, hkv):
    """Chunks from the device ring (it wraps; chunk starts off the page grid)."""
    b, layer, total = 2, 6, 3 * (w + 2 * 512 + 2 * bs) // 2 if step > 3 else 150
    q, k, v = _rand(1, b, hq, total, d), _rand(2, b, hkv, total, d), _rand(3, b, hkv, total, d)
    cache = bf.CompressedKVCache(block_size=bs, local_window_tokens=w, max_kv_size=total, max_chunk_size=512)
    for pos in range(0, total, step):
        end = min(pos + step, total)
        cache.update(k[:, :, pos:end].cuda(), v[:, :, pos:end].cuda())
        if pos == 0:
            continue
        lay, ref = _layouts(end, bs, hkv, hq // hkv, layer, "xor")
        got = bf.compressed_butterfly_attention_cached(q[:, :, pos:end].cuda(), cache, layout=lay,
                                                       local_window_tokens=w)
        ks, vs = (torch.zeros(b, hkv, lay.num_blocks, d) for _ in range(2))
        ks[:, :, :cache.summary_count], vs[:, :, :cache.summary_count] = cache.k_summary.cpu(), cache.v_summary.cpu()
        want = oa.active(q[:, :, pos:end].float(), k[:, :, :end].float(), v[:, :, :end].float(), layout=ref,
                         query_positions=torch.arange(pos, end), W=w, k_summary=ks, v_summary=vs)
        _check(got, want)
    assert step == 3 or cache.tail_capacity < total


def test_rows_without_keys_or_summaries():
    """Queries before the tail (their one summary alone), an empty pool, no summaries at all."""
    d, w, bs = 64, 100, 64
    q, k, v = _rand(1, 1, 2, 300, d), _rand(2, 1, 1, 300, d), _rand(3, 1, 1, 300, d)
    lay, _ = _layouts(500, bs, 1, 2, 1)
    pool = _rand(4, 1, 1, 1, d).cuda()
    got, _ = bf.compressed_butterfly_attention_from_cache(
        q.cuda(), k[:, :, :150].cuda(), v[:, :, :150].cuda(), pool[:, :, :1], pool[:, :, :1], layout=lay,
        query_positions=range(200, 500), local_window_tokens=w, tail_start=350, kv_len=500)
    assert torch.equal(got[0, :, :150], pool[0].expand(2, 150, d))
    o, l, m = bf.compressed_stream_attention(q.cuda(), pool[:, :, :0], pool[:, :, :0], block_size=bs, scale=0.1,
                                             routed_indices=torch.zeros(2, 5, 3, dtype=torch.int32))
    assert (o == 0).all() and (l == 0).all() and (m == -1e30).all()
    keys = k.cuda()
    core = bf.ButterflyAttentionCore(bf.compressed_butterfly_config(compressed_local_window_tokens=w,
                                                                    wayfinder_decode_backend="dense"), 0)
    want = torch.softmax(q[0, 0, :2].double() @ k[0, 0].double().T * d ** -0.5
                         + torch.tensor([[0.0] * 299 + [-math.inf], [0.0] * 300]), -1) @ v[0, 0].double()
    _check(core.attend_full(q[:, :, :2].cuda(), keys, v.cuda())[0, 0], want)


def _row(q, keys, vals, scale):
    """Softmax over an explicit key list in 64 bits."""
    s = (keys.double() @ q.double()) * scale
    return torch.softmax(s, 0) @ vals.double()


@pytest.mark.parametrize("d,groups", [(64, 1), (128, 2), (128, 4), (256, 2)])
def test_infinities_and_nans_stay_with_their_rows(d, groups):
    """An infinity or NaN in a value row reaches the queries that attend to it and no others; a NaN
    key likewise."""
    t, bs, w, layer = 400, 64, 100, 1
    hkv, hq = 1, groups
    q, k, v = _rand(4, 1, hq, t, d), _rand(5, 1, hkv, t, d), _rand(6, 1, hkv, t, d)
    v[0, 0, 130, 3] = math.inf
    v[0, 0, 207] = math.nan
    v[0, 0, 291, d - 1] = -math.inf
    k[0, 0, 350, 0] = math.nan
    lay, ref = _layouts(t, bs, hkv, groups, layer)
    ks, vs = (s for s in _summaries(k, v, bs))
    got = bf.compressed_butterfly_attention(q.cuda(), k.cuda(), v.cuda(), layout=lay, local_window_tokens=w)[0].cpu()
    rows = ref.block_neighbors[0]
    for p in range(t):
        blk = p // bs
        cut = max(0, blk * bs - w + 1)
        sel = [n for n in rows[blk].tolist() if 0 <= n < blk and (n + 1) * bs <= cut]
        lo = max(0, p - w + 1)
        keys = torch.cat([k[0, 0, lo:p + 1].float(), ks[0, 0, sel]])
        vals = torch.cat([v[0, 0, lo:p + 1].float(), vs[0, 0, sel]])
        for h in range(hq):
            want = _row(q[0, h, p].float(), keys, vals, d ** -0.5)
            g = got[0, h, p].double()
            assert torch.equal(torch.isnan(g), torch.isnan(want)) and torch.equal(torch.isinf(g), torch.isinf(want)), p
            fin = torch.isfinite(want)
            assert ((g - want)[fin].abs() <= BF16_ROUNDING * want[fin].abs() + ABS).all(), p


def _stream_check(got, want):
    o, l, m = (x.float().cpu() for x in got)
    wo, wl, wm = want
    empty = wm < -1e20
    assert torch.equal(m < -1e20, empty) and (l[empty] == 0).all()
    assert torch.allclose(m[~empty], wm[~empty], rtol=1e-5, atol=1e-5)
    # a score of size s has an fp32 error of some s 2^-22 (two or three roundings) on either side, and
    # each weight is off by that much of itself
    weight = 1e-5 + float(wm[~empty].abs().amax() if (~empty).any() else 0.0) * 2.0 ** -20
    assert torch.allclose(l[~empty], wl[~empty], rtol=weight, atol=1e-6)
    wo = wo.float()
    assert ((o - wo).abs() <= BF16_ROUNDING * wo.abs() + ABS + 5 * weight).all(), (o - wo).abs().max()


@pytest.mark.parametrize("b,hq,hkv,t,d,w,bs", [(1, 2, 1, 1, 64, 64, 128), (1, 8, 2, 700, 128, 64, 128),
                                               (2, 4, 4, 333, 64, 1, 16), (1, 4, 1, 1100, 256, 300, 64),
                                               (2, 16, 4, 2115, 128, 128, 8)])
@pytest.mark.parametrize("factor", [1.0, 40.0])
def test_streams(b, hq, hkv, t, d, w, bs, factor):
    """Window, dense and routed streams; with scores forty times as large, rows' maxima move by more
    than the kernel's rescaling threshold from group to group."""
    q, k, v = _rand(7, b, hq, t, d), _rand(8, b, hkv, t, d), _rand(9, b, hkv, t, d)
    nb = -(-t // bs)
    ks, vs = _rand(10, b, hkv, nb, d), _rand(11, b, hkv, nb, d)
    rep = lambda x: x.float().repeat_interleave(hq // hkv, dim=1)  # noqa: E731
    scale = factor * d ** -0.5
    qd, qf = q.cuda(), q.float()
    _stream_check(bf.swa_stream_attention(qd, k.cuda(), v.cuda(), n_win=w, scale=scale),
                  oa.swa_stream(qf, rep(k), rep(v), W=w, scale=scale))
    _stream_check(bf.compressed_stream_attention(qd, ks.cuda(), vs.cuda(), block_size=bs, scale=scale),
                  oa.compressed_stream(qf, rep(ks), rep(vs), block_size=bs, scale=scale))
    kcap = 3 if t > 1000 else 70
    routed = torch.randint(-2, nb + 2, (hq, nb + 1, kcap), generator=torch.Generator().manual_seed(12), dtype=torch.int32)
    _stream_check(bf.compressed_stream_attention(qd, ks.cuda(), vs.cuda(), block_size=bs, scale=scale,
                                                 routed_indices=routed.cuda()),
                  oa.compressed_stream(qf, rep(ks), rep(vs), block_size=bs, scale=scale, routed_indices=routed))


# chunk lengths, ring (max_chunk), windows and heads: the default ring with page-aligned chunks (batches
# longer than the ring, some lengths cut where slots would collide), chunks off the page grid, an
# attention window above the cache's, blocks below a page, the W <= 64 kernel with a small ring
STREAMS = [
    # d, hq, hkv, W, cache W, bs, max_chunk, chunk lengths
    (256, 16, 4, 128, 128, 128, 512, [512] * 23 + [300]),
    (128, 4, 4, 128, 128, 128, 512, [256] * 31),
    (128, 8, 2, 128, 128, 128, 320, [320, 192, 64, 320, 320, 128] * 4 + [17]),
    (64, 8, 1, 100, 64, 64, 200, [64] * 40),
    (64, 2, 2, 128, 128, 128, 512, [100, 33, 512, 3, 200, 512, 511] * 2),
    (128, 4, 2, 70, 96, 32, 256, [192] * 15),
    (128, 8, 2, 64, 64, 128, 512, [512] * 14),
    (256, 8, 2, 33, 64, 64, 256, [128] * 29 + [40]),
    (64, 4, 1, 64, 64, 128, 448, [448, 64, 384] * 6),
]


@pytest.mark.parametrize("case", STREAMS, ids=lambda c: "-".join(str(x) for x in c[:7]))
def test_stream_batches_match_single_chunks(case):
    """chunked_prefill (batched launches, updates beside attention) against one core call per chunk:
    tail, pools and counters bit for bit, and the outputs too -- up to each side's own rounding to bf16
    (2^-8 of the value and ABS) at W 65..128, where single chunks and batches may take two kernels."""
    d, hq, hkv, w, cw, bs, max_chunk, lens = case
    cfg = bf.compressed_butterfly_config(block_size=bs, compressed_local_window_tokens=w, block_partner_rule="xor")
    g = torch.Generator(device="cuda").manual_seed(5)
    chunks = [tuple(torch.randn(2, h, n, d, generator=g, device="cuda").bfloat16() for h in (hq, hkv, hkv)) for n in lens]
    caches = [bf.CompressedKVCache(block_size=bs, local_window_tokens=cw, max_kv_size=sum(lens), max_chunk_size=max_chunk)
              for _ in range(2)]
    core = bf.ButterflyAttentionCore(cfg, 5)
    got = bf.chunked_prefill(core, chunks, caches[0])
    assert core.last_profile.notes.get("native_chunk_loop")
    want = [core(*c, caches[1]) for c in chunks]
    for i, (a, b) in enumerate(zip(got, want)):
        if 64 < w <= 128:
            assert ((a.float() - b.float()).abs() <= 2 * BF16_ROUNDING * b.float().abs() + 2 * ABS).all(), i
        else:
            assert torch.equal(a, b), i
    x, y = caches
    assert (x.offset, x.tail_size, x.summary_count, x.summary_offset) == \
        (y.offset, y.tail_size, y.summary_count, y.summary_offset)
    for a, b in zip(x.get_compressed_state()[:4], y.get_compressed_state()[:4]):
        assert torch.equal(a, b)
    # the whole ring, but where the W <= 64 batches of several short chunks copy only their tails
    if w > 64 or min(a + b for a, b in zip(lens[1:], lens[2:])) > (x.tail_capacity - 128) // 2:
        assert torch.equal(x.ring_state().ring_k, y.ring_state().ring_k)
        assert torch.equal(x.ring_state().ring_v, y.ring_state().ring_v)


@pytest.mark.parametrize("w,cw,d,bs", [(1, 64, 64, 64), (65, 96, 128, 128), (65, 65, 64, 64), (40, 64, 128, 32)])
def test_streams_off_the_grid_keep_infinities_with_their_rows(w, cw, d, bs):
    """Chunks off the page grid through the native loop (each update beside the attention before it) against one
    core call per chunk, with infinities and NaN among the values: the staged rows that every query masks, down
    to three pages below a chunk, are none that the update beside writes."""
    hq, hkv, lens = 4, 2, [100] + [37, 90, 64, 11, 130, 75] * 8
    cfg = bf.compressed_butterfly_config(block_size=bs, compressed_local_window_tokens=w, block_partner_rule="xor")
    g = torch.Generator(device="cuda").manual_seed(3)
    chunks = [tuple(torch.randn(1, h, n, d, generator=g, device="cuda").bfloat16() for h in (hq, hkv, hkv)) for n in lens]
    for i in range(3, len(chunks), 5):
        chunks[i][2][0, 0, 3, 1], chunks[i][2][0, 1, 7, d - 1] = math.inf, math.nan
    caches = [bf.CompressedKVCache(block_size=bs, local_window_tokens=cw, max_kv_size=sum(lens), max_chunk_size=130)
              for _ in range(2)]
    core = bf.ButterflyAttentionCore(cfg, 2)
    got = bf.chunked_prefill(core, chunks, caches[0])
    assert core.last_profile.notes.get("native_chunk_loop")
    for i, c in enumerate(chunks):
        a, b = got[i].float(), core(*c, caches[1]).float()
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.isinf(a), torch.isinf(b)), i
        fin = torch.isfinite(b)
        assert ((a - b)[fin].abs() <= 2 * BF16_ROUNDING * b[fin].abs() + 2 * ABS).all(), i
    for a, b in zip(caches[0].get_compressed_state()[:4], caches[1].get_compressed_state()[:4]):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("d,groups", [(64, 1), (128, 2), (128, 4), (256, 2)])
def test_large_values_stay_finite(d, groups):
    """Values near bf16's largest under scores that climb by less than the rescaling threshold from group to group:
    the weighted mean is finite, and no partial sum may overflow on the way."""
    t, w, bs = 400, 200, 64
    q = torch.ones(1, groups, t, d).bfloat16()
    climb = (torch.arange(t) // 32 * 7.6 * math.log(2)) / d ** 0.5      # scores: 7.6 octaves each 32 keys
    k = climb[None, None, :, None].expand(1, 1, t, d).bfloat16()
    v = _rand(1, 1, 1, t, d)
    v[0, 0, 40::50] = 3e36 * v[0, 0, 40::50].sign()
    scale = d ** -0.5
    want = oa.swa_stream(q.double(), k.double().expand(1, groups, t, d), v.double().expand(1, groups, t, d), W=w,
                         scale=scale)[0]
    got = bf.swa_stream_attention(q.cuda(), k.cuda(), v.cuda(), n_win=w, scale=scale)[0].cpu().double()
    assert torch.isfinite(got).all()
    assert ((got - want).norm() / want.norm()).item() <= 2 ** -8
