"""CPU: when a product of 2 to 32 rows may be taken from the 4-bit codes (decoder.q4_rows_fits, less its shapes
and device): nothing follows the call's operators."""
from __future__ import annotations

import torch
import torch.nn.functional as F
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode
from torch.utils.flop_counter import FlopCounterMode

from butterfly_amd.decoder import QuantLinear, _followed, _hooked


def _layer(out_f=6, in_f=128, seed=0):
    return QuantLinear(in_f, out_f, generator=torch.Generator().manual_seed(seed))


X = torch.randn(3, 128).bfloat16()


def test_calls_that_something_follows():
    layer, seen = _layer(), []

    def call(x):
        seen.append(_followed(x, layer.weight))
        return F.linear(x, layer.weight)

    def last():
        return seen.pop()

    call(X)
    assert not last()
    torch.jit.trace(call, (X,), check_trace=False)
    assert last()
    make_fx(call)(X)
    assert last()
    with FlopCounterMode(display=False):
        call(X)
    assert last()

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        call(X)
    assert last()
    with torch.device("cpu"):      # a default device is a function mode too
        call(X)
    assert not last()
    torch.func.vmap(call)(X.unsqueeze(1))
    assert last()
    torch.func.jvp(call, (X,), (X,))
    assert last()
    call(X.clone().requires_grad_())
    assert last()
    layer.weight.requires_grad_()
    call(X)
    assert last()
    with torch.no_grad():
        call(X)
    assert not last()


def test_compiled_layers_see_the_product():
    layer = _layer()
    got = torch.compile(layer, backend="eager", fullgraph=True)(X)
    assert torch.equal(got, F.linear(X, layer.weight))


def test_hooks_and_wrappers():
    layer = _layer()
    assert not _hooked(layer)
    for register in (layer.register_forward_hook, layer.register_forward_pre_hook,
                     torch.nn.modules.module.register_module_forward_hook,
                     torch.nn.modules.module.register_module_forward_pre_hook):
        handle = register(lambda *a: None)
        assert _hooked(layer)
        handle.remove()
        assert not _hooked(layer)
    handle = layer.register_full_backward_hook(lambda *a: None)
    assert _hooked(layer)
    handle.remove()

    class Wrapped(QuantLinear):
        pass

    assert _hooked(Wrapped(128, 4))
    layer.forward = lambda x: x
    assert _hooked(layer)
