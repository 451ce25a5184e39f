"""GPU: win_attn_kernel (bf16, windows of 65 to 128 tokens, grids that fill the chip) with infinities, NaN and
values near the type's largest, against a 64-bit softmax per row.

One call of every shape here has at least 256 workgroups, from which on such windows run on that kernel; streamed
batches take it whatever their size.  Finite results are off by the output's rounding to bf16 (half an ulp, at most
2^-8 of the value) and by the weights' 16 bits and fp32 arithmetic (below 1e-5 of values of up to 5).
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
         (2, 24, 8, 1040, 256, 128, 96)]


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
            # where 3e38 takes part, its weight's 16 bits are the measure
            big = 3e38 * 2.0 ** -16 if kv == 4 and bi == 0 else 0.0
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
