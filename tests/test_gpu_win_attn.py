"""GPU: win_attn_kernel (bf16, windows of 65 to 128 tokens, grids that fill the chip) with infinities, NaN and
values near the type's largest, against a 64-bit softmax per row.

One call of every shape here has at least 256 workgroups, from which on such windows run on that kernel; streamed
batches take it whatever their size.  Finite results are off by the output's rounding to bf16 (half an ulp, at most
2^-8 of the value) and by fp32 arithmetic (below 1e-5 of values of up to 5).
"""
from __future__ import annotations

import math

import pytest
import torch

import butterfly_amd as bf
from oracle import topology as tp

pytestmark = pytest.mark.gpu

BF16_ROUNDING = 2.0 ** -8
ABS = 5e-5


def _rand(seed, *shape):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).bfloat16()


def _weighted(p, ok, v):
    """sum of p v over the keys that a row takes (ok), so that no other key's infinity reaches it."""
    finite = torch.isfinite(v)
    out = p @ torch.where(finite, v, torch.zeros_like(v))
    for r in (~finite).any(-1).nonzero()[:, 0].tolist():
        part = torch.where(finite[r], torch.zeros_like(v[r]), p[:, r:r + 1] * v[r])
        out = out + torch.where(ok[:, r:r + 1], part, torch.zeros_like(part))
    return out


def _prefill64(q, k, v, ks, vs, ref, w, bs):
    """One head's causal window and routed summaries: [t, d] in 64 bits."""
    t = q.shape[0]
    p = torch.arange(t)
    win = (p[None] <= p[:, None]) & (p[None] > p[:, None] - w)
    rows, n = ref.block_neighbors[0][p // bs], torch.arange(ks.shape[0])
    cut = (p // bs * bs - w + 1).clamp_min(0)
    far = (rows[:, :, None] == n).any(1) & (n < (p // bs)[:, None]) & ((n + 1) * bs <= cut[:, None])
    ok = torch.cat([win, far], 1)
    s = q.double() @ torch.cat([k, ks]).double().t() * q.shape[1] ** -0.5
    return _weighted(torch.softmax(s.masked_fill(~ok, -math.inf), -1), ok, torch.cat([v, vs]).double())


# b, hq, hkv, t, d, bs, W: groups of 1, 2 and 3 heads (one and two heads a wave, one of them empty), four heads a
# workgroup at d = 256, blocks of half a page, lengths off the page and the 16-row tile
CASES = [(4, 8, 8, 533, 64, 64, 65), (4, 16, 8, 530, 64, 32, 128), (4, 8, 8, 560, 128, 64, 100),
         (3, 24, 8, 700, 128, 128, 128), (4, 16, 8, 521, 128, 64, 127), (4, 8, 8, 530, 256, 64, 128),
         (2, 24, 8, 1040, 256, 128, 96), (2, 32, 8, 530, 256, 64, 128)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x) for x in c))
def test_infinities_and_nans_stay_with_their_rows(case):
    b, hq, hkv, t, d, bs, w = case
    g = hq // hkv
    assert ((t - 1) // 64 + 1) * b * hkv * (1 if g == 1 else (g + 1) // 2) >= 256
    q, k, v = _rand(1, b, hq, t, d), _rand(2, b, hkv, t, d), _rand(3, b, hkv, t, d)
    # (0, 0): one value a row, in the window's first and last tiles and inside blocks that are summarised later
    v[0, 0, 3, 0], v[0, 0, 130, 5], v[0, 0, 200, d - 1], v[0, 0, 333, 17] = math.inf, -math.inf, math.inf, math.nan
    v[0, 1, 70], v[0, 1, 410, ::2], v[0, 1, 411, 1::2] = math.nan, math.inf, -math.inf      # whole rows
    k[0, 2, 150, 4], k[0, 2, 320, 1] = math.nan, math.inf
    v[0, 3, 255, 3], v[0, 3, 256, 3] = math.inf, -math.inf                 # both signs for some rows: NaN
    v[0, 4, 100, 7] = 3e38
    v[b - 1, hkv - 1, t - 1, 2] = -math.inf                               # the newest token
    kw = dict(seq_len=t, block_size=bs, num_key_value_heads=hkv, num_key_value_groups=g, layer_idx=2,
              local_window_blocks=1, sink_count=1, partner_count=1, partner_rule="xor")
    ref = tp.build_layout(**kw)
    kd, vd = k.cuda(), v.cuda()
    ks, vs = (s.cpu() for s in bf.block_mean_summaries(kd, seq_len=t, block_size=bs, num_blocks=-(-t // bs), x2=vd))
    got = bf.compressed_butterfly_attention(q.cuda(), kd, vd, layout=bf.build_block_butterfly_layout(**kw),
                                            local_window_tokens=w)[0].cpu().double()
    heads = [(0, kv) for kv in range(5)] + [(b - 1, hkv - 1), (1, 0)]
    seen = 0
    for bi, kv in heads:
        for h in range(kv * g, kv * g + g):
            want, out = _prefill64(q[bi, h], k[bi, kv], v[bi, kv], ks[bi, kv], vs[bi, kv], ref, w, bs), got[bi, h]
            assert torch.equal(torch.isnan(out), torch.isnan(want)), (bi, h)
            assert torch.equal(torch.isposinf(out), torch.isposinf(want)), (bi, h)
            assert torch.equal(torch.isneginf(out), torch.isneginf(want)), (bi, h)
            fin = torch.isfinite(want)
            # where 3e38 takes part, its weight's fp32 rounding is the measure (scores of up to 8: below 2^-20)
            big = 3e38 * 2.0 ** -20 if kv == 4 and bi == 0 else 0.0
            room = BF16_ROUNDING * want.abs() + ABS + big * (torch.arange(d) == 7)
            assert ((out - want).abs() <= room)[fin].all(), (bi, h)
            seen += int((~fin).sum())
    assert seen > 1000


@pytest.mark.parametrize("d,hq,hkv,bs,lens", [(64, 6, 2, 64, [128] * 12), (128, 4, 4, 128, [512] * 5 + [77]),
                                              (256, 8, 2, 128, [256] * 7 + [130]), (128, 6, 2, 64, [100, 37, 90] * 5)])
def test_streamed_batches_keep_them_too(d, hq, hkv, bs, lens):
    """chunked_prefill at W = 128: pages from the chunk inputs and from the ring, positions that do not exist beside rows that hold an infinity."""
    t, w = sum(lens), 128
    q, k, v = _rand(4, 1, hq, t, d), _rand(5, 1, hkv, t, d), _rand(6, 1, hkv, t, d)
    ends = torch.tensor(lens).cumsum(0).tolist()
    for i, e in enumerate(ends[:-1]):             # on both sides of the chunks' borders
        v[0, i % hkv, e - 1, i % d], v[0, (i + 1) % hkv, e, (i + 3) % d] = math.inf, math.nan
    k[0, 0, ends[2] + 1, 0] = math.nan
    cfg = bf.compressed_butterfly_config(block_size=bs, compressed_local_window_tokens=w, block_partner_rule="xor")
    core = bf.ButterflyAttentionCore(cfg, 3)
    cache = bf.CompressedKVCache(block_size=bs, local_window_tokens=w, max_kv_size=t, max_chunk_size=512)
    starts = [0] + ends[:-1]
    chunks = [tuple(x[:, :, s:e].cuda().contiguous() for x in (q, k, v)) for s, e in zip(starts, ends)]
    got = bf.chunked_prefill(core, chunks, cache)
    assert core.last_profile.notes.get("native_chunk_loop")
    pk, pv, seen = cache._pool_k.cpu(), cache._pool_v.cpu(), 0
    for c in range(1, len(lens)):
        s, e = starts[c], ends[c]
        rows = tp.build_layout(seq_len=e, block_size=bs, num_key_value_heads=hkv, num_key_value_groups=hq // hkv,
                               layer_idx=3, local_window_blocks=1, sink_count=1, partner_count=1,
                               partner_rule="xor").block_neighbors[0]
        nsum = max(0, (e - w) // bs)
        p, n, at = torch.arange(s, e), torch.arange(nsum), torch.arange(e)
        win = (at[None] <= p[:, None]) & (at[None] > p[:, None] - w)
        far = (rows[p // bs][:, :, None] == n).any(1) & (n < (p // bs)[:, None]) & \
            ((n + 1) * bs <= (p - w + 1).clamp_min(0)[:, None])
        ok = torch.cat([win, far], 1)
        for h in range(hq):
            kv = h // (hq // hkv)
            sc = q[0, h, s:e].double() @ torch.cat([k[0, kv, :e], pk[0, kv, :nsum]]).double().t() * d ** -0.5
            want = _weighted(torch.softmax(sc.masked_fill(~ok, -math.inf), -1), ok,
                             torch.cat([v[0, kv, :e], pv[0, kv, :nsum]]).double())
            out = got[c][0, h].cpu().double()
            assert torch.equal(torch.isnan(out), torch.isnan(want)) and torch.equal(torch.isinf(out), torch.isinf(want)), (c, h)
            fin = torch.isfinite(want)
            assert ((out - want).abs() <= BF16_ROUNDING * want.abs() + ABS)[fin].all(), (c, h)
            seen += int((~fin).sum())
    assert seen > 100


# kind, hq, hkv, t, d, W: win_attn_kernel with one and two heads a wave and four a workgroup, page_attn_kernel (small
# grids, W above 128) in its splits, the window stream, and the dense summary stream (every earlier block of 16)
WEIGHTS = [("call", 4, 4, 4160, 64, 128), ("call", 8, 4, 4160, 128, 100), ("call", 12, 4, 4160, 256, 128),
           ("call", 2, 2, 1000, 128, 128), ("call", 8, 2, 1000, 256, 200), ("call", 16, 4, 4160, 128, 256),
           ("call", 2, 1, 9000, 64, 256), ("window", 8, 4, 4160, 128, 128), ("window", 4, 4, 2000, 64, 64),
           ("dense", 8, 2, 2000, 128, 1), ("dense", 4, 4, 2000, 64, 1)]


@pytest.mark.parametrize("kind,hq,hkv,t,d,w", WEIGHTS)
def test_weights_keep_fp32_precision(kind, hq, hkv, t, d, w):
    """Values that cancel under a row's weights leave the weights' own error: some queries with windows apart, each
    with four keys chosen so that the weighted sum of every column is next to zero.  Scores near zero keep an fp32
    weight within about 2^-23 of itself, and sums of random sign come to 2^-22.5 of size = sqrt(sum (p v)^2); weights
    of 16 bits miss by 2^-19.5 of size (rms)."""
    g, bs = hq // hkv, 16 if kind == "dense" else 128
    q, k, v = _rand(1, 1, hq, t, d) * 0.05, _rand(2, 1, hkv, t, d), _rand(3, 1, hkv, t, d)
    n = t // bs if kind == "dense" else 0
    ks, vs = _rand(4, 1, hkv, max(n, 1), d), _rand(5, 1, hkv, max(n, 1), d)
    keys, vals, rows = (ks, vs, [t - 1]) if kind == "dense" else (k, v, range(w + 70, t, w + 113))
    picked = []
    for kv in range(hkv):
        for i, r in enumerate(rows):
            h = kv * g + i % g
            lo, hi = (0, r // bs) if kind == "dense" else (r - w + 1, r + 1)
            p = torch.softmax((keys[0, kv, lo:hi].double() @ q[0, h, r].double()) * d ** -0.5, -1)[:, None]
            x = vals[0, kv, lo:hi].double()
            for key in (hi - lo) * torch.tensor([1, 3, 6, 8]) // 9:
                x[key] = 0
                x[key] = (-(p * x).sum(0) / p[key]).bfloat16().double()
            vals[0, kv, lo:hi] = x.bfloat16()
            picked.append((h, r, (p * x).sum(0), (p * x).pow(2).sum(0).sqrt()))
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    if kind == "call":
        lay = bf.build_block_butterfly_layout(seq_len=t, block_size=bs, num_key_value_heads=hkv, num_key_value_groups=g,
                                              layer_idx=0, local_window_blocks=0, sink_count=0, partner_count=0,
                                              partner_rule="xor")      # no summaries
        got = bf.compressed_butterfly_attention(qd, kd, vd, layout=lay, local_window_tokens=w)[0]
    elif kind == "window":
        got = bf.swa_stream_attention(qd, kd, vd, n_win=w, scale=d ** -0.5)[0]
    else:
        got = bf.compressed_stream_attention(qd, ks.cuda(), vs.cuda(), block_size=bs, scale=d ** -0.5)[0]
    got = got[0].cpu().double()
    worst = max(((got[h, r] - want).abs() - BF16_ROUNDING * want.abs()).div(size).max().item()
                for h, r, want, size in picked)
    assert worst <= 2.0 ** -20
