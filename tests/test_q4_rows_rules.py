"""CPU: when a product of 2 to 32 rows may be taken from the 4-bit codes (decoder.q4_rows_fits, less its shapes
and device): nothing follows the call's operators, and ``weight`` still is what the codes say."""
from __future__ import annotations

import copy
import pickle

import pytest
import torch
import torch.nn.functional as F
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode
from torch.utils.flop_counter import FlopCounterMode

from butterfly_amd.decoder import Decoder, DecoderConfig, QuantLinear, _followed, _hooked


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


def _replace_functionally(layer):
    with torch.no_grad():
        got = []
        layer.register_forward_pre_hook(lambda m, a: got.append(m.codes_hold()))
        torch.func.functional_call(layer, {"weight": layer.weight.clone()}, (X,))
        assert layer.codes_hold()
    if not got[0]:
        layer._bound = None


EDITS = {
    "in place": lambda layer: layer.weight.mul_(2),
    "one row through a view": lambda layer: layer.weight[1].add_(1),
    "another tensor": lambda layer: setattr(layer, "weight", layer.weight.clone()),
    "other data": lambda layer: setattr(layer.weight, "data", layer.weight.clone()),
    "codes in place": lambda layer: layer.packed.zero_(),
    "pairs in place": lambda layer: layer.scale_bias.mul_(2),
    "under inference": lambda layer: torch.inference_mode()(lambda: layer.weight.mul_(2))(),
    "functional_call": _replace_functionally,
}


@pytest.mark.parametrize("edit", EDITS)
def test_edits_end_it(edit):
    layer = _layer()
    assert layer.codes_hold()
    EDITS[edit](layer)
    assert not layer.codes_hold()


def test_fused_layers_share_their_edits():
    a, b = _layer(4), _layer(8, seed=1)
    both = QuantLinear.fuse_rows(a, b)
    assert a.codes_hold() and b.codes_hold() and both.codes_hold()
    b.weight.mul_(2)
    assert not both.codes_hold()
    c, d = _layer(4), _layer(4)
    d.weight.mul_(2)
    assert not QuantLinear.fuse_rows(c, d).codes_hold()


def test_copies_moves_and_loads_keep_it():
    layer = _layer()
    for same in (copy.deepcopy(layer), pickle.loads(pickle.dumps(layer)), copy.deepcopy(layer).to(torch.bfloat16)):
        assert same.codes_hold() and torch.equal(same.weight, layer.weight)
    other = _layer(seed=5)
    other.load_state_dict(layer.state_dict())
    assert other.codes_hold() and torch.equal(other.packed, layer.packed)
    with torch.inference_mode():
        made = _layer()
    assert made.codes_hold()
    # what an edit ended stays ended
    layer.weight[0, 0] += 1
    other.load_state_dict(layer.state_dict())
    assert not other.codes_hold()
    for edited in (copy.deepcopy(layer), pickle.loads(pickle.dumps(layer)), copy.deepcopy(layer).to(torch.bfloat16)):
        assert not edited.codes_hold()


def test_tensors_without_values():
    """Building, moving and loading under FakeTensorMode or on the meta device."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    with FakeTensorMode():
        layer = QuantLinear(128, 4, weight=torch.randn(4, 128))
        layer.to(torch.float32).load_state_dict(layer.state_dict())
        assert not layer.codes_hold()
    assert _layer().to("meta").weight.is_meta


def test_compiled_layers_see_the_product():
    layer = _layer()
    got = torch.compile(layer, backend="eager", fullgraph=True)(X)
    assert torch.equal(got, F.linear(X, layer.weight))


def test_the_embedding_counts_the_head_weights_edits():
    cfg = DecoderConfig(vocab_size=64, hidden_size=128, num_layers=0)
    model = Decoder(cfg, device="cpu")
    assert model.embed_tokens.data_ptr() == model.lm_head.weight.data_ptr() and model.lm_head.codes_hold()
    with torch.no_grad():
        model.embed_tokens[3].zero_()
    assert not model.lm_head.codes_hold()


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
