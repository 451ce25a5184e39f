"""GPU: the q/k norm and RoPE launch that reads its table row at a device position."""
from __future__ import annotations

import pytest
import torch

from butterfly_amd.decoder import Attention, DecoderConfig, RopeTable, rope_cos_sin

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,b,pos", [(128, 1, 0), (128, 8, 41), (256, 3, 99)])
@pytest.mark.parametrize("pad", [0, 3])
def test_table_row_equals_selected_rows(d, b, pos, pad):
    """Same arithmetic on the same row: bit for bit, also from tables whose base is not 16-byte aligned."""
    cfg = DecoderConfig(hidden_size=512, num_heads=4, num_kv_heads=2, head_dim=d)
    attn = Attention(cfg, generator=torch.Generator("cuda").manual_seed(1), device="cuda")
    qkv = torch.randn(b, 1, 8 * d, generator=torch.Generator().manual_seed(2)).bfloat16().cuda()
    tabs = []
    for t in rope_cos_sin(torch.arange(100), d, 1e6):
        buf = torch.zeros(100 * d + pad, device="cuda")
        buf[pad:] = t.reshape(-1).cuda()
        tabs.append(buf[pad:].view(100, d))
    table = RopeTable(*tabs, torch.tensor([pos], device="cuda"))
    assert table.fits(qkv, d)
    for got, want in zip(attn.heads(qkv, None, table), attn.heads(qkv, None, table.rows())):
        assert torch.equal(got, want)


def test_position_off_the_table_is_nan():
    cfg = DecoderConfig(hidden_size=512, num_heads=4, num_kv_heads=2, head_dim=128)
    attn = Attention(cfg, generator=torch.Generator("cuda").manual_seed(1), device="cuda")
    qkv = torch.ones(2, 1, 1024, dtype=torch.bfloat16, device="cuda")
    cos, sin = (t.cuda().contiguous() for t in rope_cos_sin(torch.arange(10), 128, 1e6))
    for pos in (-1, 10):
        q, k, v = attn.heads(qkv, None, RopeTable(cos, sin, torch.tensor([pos], device="cuda")))
        assert torch.isnan(q).all() and torch.isnan(k).all() and (v == 1).all()
