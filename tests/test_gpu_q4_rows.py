"""GPU: products of 2 to 32 rows from the 4-bit codes (bfly_q4_rows, bfly_q4_rows_silu).

Against 64-bit sums over w = code * scale + bias: the output's rounding to bf16 (at most 2^-8 of the value),
and fp32 sums of terms x (16 + code) scale and x (bias - 16 scale), whose error is below
2^-20 of the sum of their magnitudes (four roundings of 2^-24 on each, few-fold accumulation).
"""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from butterfly_amd import _native
from butterfly_amd._device import stream_of
from butterfly_amd.decoder import MLP, Decoder, DecoderConfig, QuantLinear, q4_rows, q4_rows_fits, q4_rows_silu

pytestmark = pytest.mark.gpu


def _layer(out_f, in_f, seed):
    g = torch.Generator().manual_seed(seed)
    # a mean away from zero: scale and bias parts that do not cancel
    return QuantLinear(in_f, out_f, weight=torch.randn(out_f, in_f, generator=g) * 0.05 + 0.01).cuda()


def _reference(x, layer):
    codes = torch.stack([layer.packed & 0xF, layer.packed >> 4], -1).flatten(1).double().view(layer.out_features, -1, 64)
    s, b = layer.scale.double().unsqueeze(-1), layer.bias.double().unsqueeze(-1)
    want = x.double() @ (codes * s + b).flatten(1).t()
    size = x.double().abs() @ ((16 + codes) * s.abs() + (b - 16 * s).abs()).flatten(1).t()
    return want, size * 2.0 ** -20


# tiles that end short, one run of 256 inputs (waves without work), runs that do not divide by the
# waves, the wide form (from 16384 outputs) with its last tile short and with its larger LDS
@pytest.mark.parametrize("rows,out_f,in_f", [(2, 1, 256), (3, 17, 512), (8, 3072, 2048), (16, 100, 6144), (16, 48, 2304),
                                             (17, 33, 256), (32, 2048, 2048), (32, 16400, 512), (2, 16385, 256),
                                             (5, 16400, 2048), (16, 20000, 4096), (16, 16384, 4352), (9, 40001, 768)])
def test_rows(rows, out_f, in_f):
    layer = _layer(out_f, in_f, rows + out_f)
    x = torch.randn(rows, in_f, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    assert q4_rows_fits(x, layer)
    want, tol = _reference(x, layer)
    got = layer(x.view(rows, 1, in_f)).view(rows, out_f).double()
    assert ((got - want).abs() <= want.abs() * 2.0 ** -8 + tol).all(), (got - want).abs().max()


@pytest.mark.parametrize("rows", [2, 16, 17, 32])
@pytest.mark.parametrize("f,in_f", [(6144, 2048), (100, 512)])
def test_silu(rows, f, in_f):
    """SiLU(gate) * up in the product's launch equals bfly_silu_mul over the two products, but for
    the products' summation order (two and four tiles add the same parts in the same order)."""
    gate_up = _layer(2 * f, in_f, f)
    x = torch.randn(rows, in_f, generator=torch.Generator().manual_seed(2)).bfloat16().cuda()
    gu = q4_rows(x, gate_up)
    want = torch.empty(rows, f, dtype=torch.bfloat16, device="cuda")
    _native.call("bfly_silu_mul", gu.data_ptr(), gu.data_ptr() + 2 * f, rows, f, 2 * f, want.data_ptr(), stream_of(x))
    got = q4_rows_silu(x, gate_up)
    # one bf16 step of gate, up or the product where the splits over waves differ
    assert ((got.float() - want.float()).abs() <= want.float().abs() * 2.0 ** -6 + 1e-6).all()
    assert (got == want).float().mean() > 0.97


def test_what_takes_the_codes():
    layer = _layer(64, 256, 3)
    x = torch.randn(4, 256, device="cuda").bfloat16()
    assert q4_rows_fits(x, layer) and not q4_rows_fits(x[:1], layer)
    assert not q4_rows_fits(x.float(), layer) and not q4_rows_fits(x.repeat(9, 1), layer)
    assert not q4_rows_fits(x, _layer(64, 192, 4)) and not q4_rows_fits(x.cpu(), layer)
    # gradients and transforms go through the GEMM
    xg = x.clone().requires_grad_()
    assert not q4_rows_fits(xg, layer)
    layer(xg).float().sum().backward()
    assert torch.allclose(xg.grad.float(), layer.weight.float().sum(0).expand(4, -1), rtol=2 ** -7, atol=1e-3)
    with torch.no_grad():
        assert q4_rows_fits(xg, layer)
    y = torch.func.vmap(layer)(x.view(2, 2, 256)).view(4, 64)
    assert torch.equal(y, F.linear(x.view(2, 2, 256), layer.weight).view(4, 64))
    # strided and unaligned rows
    wide = torch.randn(4, 520, device="cuda").bfloat16()
    want, tol = _reference(wide[:, 3:259], layer)
    got = layer(wide[:, 3:259]).double()
    assert ((got - want).abs() <= want.abs() * 2.0 ** -8 + tol).all()
    with pytest.raises(ValueError, match="rows"):
        q4_rows(torch.zeros(33, 256, dtype=torch.bfloat16, device="cuda"), layer)


def test_mlp_rows_match_one_by_one():
    cfg = DecoderConfig(hidden_size=512, intermediate_size=1024)
    mlp = MLP(cfg, generator=torch.Generator(device="cuda").manual_seed(0), device="cuda")
    x = torch.randn(6, 1, 512, device="cuda").bfloat16()
    got = mlp(x)
    one = torch.cat([mlp(r.unsqueeze(0)) for r in x])
    # the rows' inner activations may differ by a bf16 step where the sums' order rounds differently
    assert ((got - one).float().norm() / one.float().norm()).item() <= 2 ** -8


@pytest.mark.parametrize("rows,out_f,in_f", [(2, 40, 256), (16, 100, 2304), (17, 33, 1024), (32, 16400, 512),
                                             (5, 16400, 2048), (16, 16400, 4096)])
def test_infinities_and_large_values(rows, out_f, in_f):
    """An infinity or NaN in a row gives what the product over ``weight`` gives, and a row of values near the type's
    largest stays finite where that product is; the other rows do not change."""
    layer = _layer(out_f, in_f, 5)
    x = torch.randn(rows, in_f, generator=torch.Generator().manual_seed(6)).bfloat16().cuda()
    plain = layer(x)
    at = 70 % in_f
    bad = x.clone()
    bad[0, at], bad[1, at] = float("inf"), 3e38         # one value: 3e38 w is finite, 3e38 (16 + code) is not
    if rows > 5:
        bad[3, 1], bad[3, in_f - 1], bad[4, at], bad[rows - 1, 9] = float("inf"), float("inf"), float("-inf"), float("nan")
    got, want = layer(bad).double(), bad.double() @ layer.weight.double().t()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isposinf(got), torch.isposinf(want))
    assert torch.equal(torch.isneginf(got), torch.isneginf(want)) and torch.isinf(got[0]).any()
    fin = torch.isfinite(want[1])
    # 3e38 times a weight rounded to bf16 (2^-9 of it) or not, and the output's own rounding
    assert fin.all() and ((got[1] - want[1]).abs() <= 2.0 ** -7 * want[1].abs() + 2.0 ** -20 * 3e38).all()
    same = [r for r in range(rows) if bool((bad[r] == x[r]).all())]
    assert torch.equal(got[same], plain[same].double())


def test_silu_infinities():
    gate_up = _layer(200, 512, 7)
    x = torch.randn(4, 512, generator=torch.Generator().manual_seed(8)).bfloat16().cuda()
    x[0, 3], x[2, 500] = float("inf"), float("-inf")
    gu = F.linear(x, gate_up.weight)
    want, got = F.silu(gu[:, :100]) * gu[:, 100:], q4_rows_silu(x, gate_up)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))


def _few(layer, n=4):
    return torch.randn(n, layer.in_features, generator=torch.Generator().manual_seed(9)).bfloat16().cuda()


def test_traced_layers_record_the_product():
    layer = _layer(48, 256, 11)
    x = _few(layer)
    traced = torch.jit.trace(layer, (x,), check_trace=False)
    other = torch.flip(x, (0,))
    assert torch.equal(traced(other), F.linear(other, layer.weight))


def test_weight_gradients_edits_and_autocast():
    layer = _layer(48, 256, 12)
    x = _few(layer)
    with torch.autocast("cuda", dtype=torch.float16):
        assert layer(x).dtype == torch.float16
    layer.weight.requires_grad_()
    layer(x).float().sum().backward()
    assert torch.allclose(layer.weight.grad.float(), x.float().sum(0).expand(48, -1), rtol=2 ** -7, atol=1e-3)
    layer.weight.requires_grad_(False)
    assert q4_rows_fits(x, layer)
    layer.weight[7].zero_()
    assert (layer(x)[:, 7] == 0).all() and torch.equal(layer(x), F.linear(x, layer.weight))


def test_mlp_hooks_fire():
    cfg = DecoderConfig(hidden_size=512, intermediate_size=1024)
    mlp = MLP(cfg, generator=torch.Generator(device="cuda").manual_seed(0), device="cuda")
    x, seen = torch.randn(6, 1, 512, device="cuda").bfloat16(), []
    plain = mlp(x)
    handle = mlp.gate_up.register_forward_hook(lambda m, a, out: seen.append(out.shape))
    got = mlp(x)
    handle.remove()
    assert seen == [(6, 1, 2048)]
    assert ((got - plain).float().norm() / plain.float().norm()).item() <= 2 ** -8


def test_logits_follow_the_embedding():
    cfg = DecoderConfig(vocab_size=512, hidden_size=256, num_layers=0)
    model = Decoder(cfg, device="cuda")
    h = torch.randn(4, 256, device="cuda").bfloat16()
    before = model._logits(h)
    with torch.no_grad():
        model.embed_tokens[5].zero_()
    after = model._logits(h)
    assert (after[:, 5] == 0).all() and ((after - before)[:, :5].float().abs() <= 2 ** -6 * before[:, :5].float().abs() + 1e-2).all()
