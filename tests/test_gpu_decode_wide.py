"""GPU: the fused one-token step for bf16 windows of 65 to 128 tokens.

Each step is compared with a 64-bit softmax over the same bf16 rows and the device's own summaries:
what remains is the output's rounding to bf16 (half an ulp, at most 2^-8 of the value) and fp32
arithmetic on scores and weights (about 1e-6 relative, times values of up to 5).  The buffers must be
those that ``update`` leaves, and infinities and NaN reach the rows that attend to them as they would
in the softmax.
"""
from __future__ import annotations

import math

import pytest
import torch

import butterfly_amd as bf
from butterfly_amd import _native
from oracle import topology as tp

pytestmark = pytest.mark.gpu

BF16_ROUNDING = 2.0 ** -8
ABS = 5e-5


def _rand(seed, *shape):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).bfloat16()


# b, hq, hkv, d, bs, W, prompt, steps: the window's edges, GQA groups of 1, 3, 4 and 20 (two head
# passes), prompts shorter than the window, steps that complete blocks and wrap the ring
CASES = [
    (1, 16, 4, 128, 128, 128, 380, 140),
    (2, 3, 1, 128, 64, 65, 3, 150),
    (3, 4, 4, 64, 128, 127, 250, 20),
    (1, 20, 1, 64, 64, 100, 500, 70),
    (1, 8, 2, 256, 128, 128, 300, 90),
    (2, 20, 1, 256, 256, 96, 700, 70),
]


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("case", CASES)
def test_wide_steps(case, special, monkeypatch):
    b, hq, hkv, d, bs, w, prompt, steps = case
    total, g = prompt + steps, hq // hkv
    q, k, v = _rand(1, b, hq, total, d), _rand(2, b, hkv, total, d), _rand(3, b, hkv, total, d)
    if special:
        at = max(prompt - 20, 0)
        v[0, 0, at, 3], v[0, 0, at + 1, d - 1] = math.inf, -math.inf
        v[0, 0, prompt + 5, 7] = math.nan
        v[0, 0, prompt + 6, 20] = 3e38
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    kw = dict(block_size=bs, local_window_tokens=w, max_kv_size=total)
    cache, plain = bf.CompressedKVCache(**kw), bf.CompressedKVCache(**kw)
    for c in (cache, plain):
        c.update(kd[:, :, :prompt], vd[:, :, :prompt])
    calls, native = [], _native.call
    monkeypatch.setattr(_native, "call", lambda name, *a: (calls.append(name), native(name, *a))[1])
    for pos in range(prompt, total):
        lkw = dict(seq_len=pos + 1, block_size=bs, num_key_value_heads=hkv, num_key_value_groups=g, layer_idx=3,
                   local_window_blocks=1, sink_count=1, partner_count=1, partner_rule="causal_shift")
        s = slice(pos, pos + 1)
        calls.clear()
        got = cache.update_and_attend(qd[:, :, s], kd[:, :, s], vd[:, :, s],
                                      layout=bf.build_block_butterfly_layout(**lkw), local_window_tokens=w)
        assert "bfly_decode_wide" in calls and "bfly_attend_cache" not in calls
        plain.update(kd[:, :, s], vd[:, :, s])
        if pos % 7 and pos < total - 3:
            continue
        blk, lo, cut = pos // bs, max(0, pos - w + 1), max(0, pos - w + 1)
        row = tp.build_layout(**lkw).block_neighbors[0][blk].tolist()
        sel = [n for n in row if 0 <= n < blk and n < cache.summary_count and (n + 1) * bs <= cut]
        pk, pv = cache._pool_k.cpu(), cache._pool_v.cpu()
        keys = torch.cat([k[:, :, lo:pos + 1], pk[:, :, sel]], 2).double().repeat_interleave(g, 1)
        vals = torch.cat([v[:, :, lo:pos + 1], pv[:, :, sel]], 2).double().repeat_interleave(g, 1)
        p = torch.softmax((keys @ q[:, :, pos].double()[..., None])[..., 0] * d ** -0.5, -1)
        want, out = (p[..., None] * vals).sum(2), got[:, :, 0].cpu().double()
        assert torch.equal(torch.isnan(out), torch.isnan(want)), pos
        assert torch.equal(torch.isinf(out), torch.isinf(want)), pos
        fin = torch.isfinite(want)
        assert ((out - want)[fin].abs() <= BF16_ROUNDING * want[fin].abs() + ABS).all(), pos
    for a in ("_ring_k", "_ring_v", "_pool_k", "_pool_v"):
        x, y = getattr(cache, a), getattr(plain, a)
        n = cache.summary_count if "pool" in a else min(total, cache.tail_capacity)
        assert torch.equal(x[:, :, :n].view(torch.int16), y[:, :, :n].view(torch.int16)), a


def test_general_path_calls_stay_accepted():
    """fp32, windows above 128 and a scale that is not positive keep the general path."""
    for dtype, w, scale in ((torch.float32, 100, None), (torch.bfloat16, 129, None), (torch.bfloat16, 100, -0.1)):
        q, k = _rand(5, 1, 4, 301, 64).to(dtype), _rand(6, 1, 2, 301, 64).to(dtype)
        cache = bf.CompressedKVCache(block_size=64, local_window_tokens=w, max_kv_size=400)
        cache.update(k[:, :, :300].cuda(), k[:, :, :300].cuda())
        lay = bf.build_block_butterfly_layout(seq_len=301, block_size=64, num_key_value_heads=2,
                                              num_key_value_groups=2, layer_idx=0, local_window_blocks=1,
                                              sink_count=1, partner_count=1, partner_rule="xor")
        out = cache.update_and_attend(q[:, :, 300:].cuda(), k[:, :, 300:].cuda(), k[:, :, 300:].cuda(), layout=lay,
                                      local_window_tokens=w, scale=scale)
        assert torch.isfinite(out).all()


def test_heads_that_do_not_group_are_refused_after_the_append():
    """Three query heads over two: refused, and the token is in the cache, as on the general path."""
    k = _rand(6, 1, 2, 301, 64)
    lay = bf.build_block_butterfly_layout(seq_len=301, block_size=64, num_key_value_heads=2, num_key_value_groups=2,
                                          layer_idx=0, local_window_blocks=1, sink_count=1, partner_count=1,
                                          partner_rule="xor")
    caches = []
    for w in (100, 129):      # the fused step's windows, the general path's
        cache = bf.CompressedKVCache(block_size=64, local_window_tokens=128, max_kv_size=400)
        cache.update(k[:, :, :300].cuda(), k[:, :, :300].cuda())
        with pytest.raises(ValueError, match="head"):
            cache.update_and_attend(_rand(7, 1, 3, 1, 64).cuda(), k[:, :, 300:].cuda(), k[:, :, 300:].cuda(), layout=lay,
                                    local_window_tokens=w)
        caches.append(cache)
    for a, b in zip(caches[0].get_compressed_state()[:4], caches[1].get_compressed_state()[:4]):
        assert torch.equal(a, b)
    assert caches[0].offset == caches[1].offset == 301


@pytest.mark.parametrize("d", [64, 128, 256])
def test_weights_keep_fp32_precision(d):
    """Values that cancel under the weights leave the weights' own error: four window rows of each column are
    chosen so that the weighted sum is next to zero.  Scores near zero keep an fp32 weight within about 2^-24 of
    itself, and the sums of random sign come to 2^-23 of size = sqrt(sum (p v)^2); weights of 16 bits miss by
    2^-19.5 of size (rms)."""
    h, w, bs, prompt = 4, 128, 128, 400
    q, k, v = _rand(1, 1, h, 1, d) * 0.05, _rand(2, 1, h, prompt + 1, d), _rand(3, 1, h, prompt + 1, d).double()
    keys = k[0].double()[:, prompt - w + 1:]
    kw = dict(seq_len=prompt + 1, block_size=bs, num_key_value_heads=h, num_key_value_groups=1, layer_idx=0,
              local_window_blocks=0, sink_count=0, partner_count=0, partner_rule="xor")     # no summaries
    p = torch.softmax((keys @ q[0].double().transpose(1, 2))[..., 0] * d ** -0.5, -1)[..., None]    # [h, w, 1]
    vals = v[0, :, prompt - w + 1:]                                                                # a view
    for row in (20, 50, 90, 120):
        vals[:, row] = 0
        vals[:, row] = (-(p * vals).sum(1) / p[:, row]).bfloat16().double()
    cache = bf.CompressedKVCache(block_size=bs, local_window_tokens=w, max_kv_size=512)
    kd, vd = k.cuda(), v.bfloat16().cuda()
    cache.update(kd[:, :, :prompt], vd[:, :, :prompt])
    got = cache.update_and_attend(q.cuda(), kd[:, :, prompt:], vd[:, :, prompt:],
                                  layout=bf.build_block_butterfly_layout(**kw), local_window_tokens=w)
    want, size = (p * vals).sum(1), (p * vals).pow(2).sum(1).sqrt()
    off = (got[0, :, 0].cpu().double() - want).abs() - 2.0 ** -8 * want.abs()
    assert (off / size).max() <= 2.0 ** -20
