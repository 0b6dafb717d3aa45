"""Where swiglu may be part of the gate_up product (CPU: the product is
stood in for)."""
import pytest
import torch
import torch.nn as nn

import llmlb_amd.ops as ops
from llmlb_amd.models.llama import LlamaConfig, LlamaForCausalLM
from llmlb_amd.parallel import tp


@pytest.fixture
def layer(monkeypatch):
    """(model, names of the products with an activation that ran)"""
    ran = []

    def stand_in(x, weight, act, up=0):
        ran.append(act)
        z = torch.nn.functional.linear(x, weight)
        return torch.nn.functional.silu(z[:, :up]) * z[:, up:]

    monkeypatch.setattr(ops, "linear_act", stand_in)
    cfg = LlamaConfig.tiny()
    return LlamaForCausalLM(cfg, dtype=torch.float32, device="cpu",
                            seed=3), ran


def _run(model):
    cfg = model.cfg
    g = torch.Generator().manual_seed(1)
    attn = torch.randn(3, cfg.q_heads, cfg.head_dim, generator=g)
    return model.layer_attn_epilogue(
        0, attn, torch.randn(3, cfg.hidden, generator=g))[0]


def test_plain_module_is_fused(layer):
    model, ran = layer
    _run(model)
    assert ran == ["swiglu"]


def test_bias_is_added(layer):
    model, ran = layer
    up = model.layers_[0].gate_up
    before = _run(model)
    up.bias = nn.Parameter(torch.full((up.out_local,), 0.5),
                           requires_grad=False)
    ran.clear()
    after = _run(model)
    assert ran == [] and not torch.allclose(before, after)


@pytest.mark.parametrize("register", [
    lambda m, f: m.register_forward_hook(lambda mod, i, o: f(o)),
    lambda m, f: m.register_forward_pre_hook(lambda mod, i: f(i[0])),
    lambda m, f: nn.modules.module.register_module_forward_hook(
        lambda mod, i, o: f(o) if mod is m else None)],
    ids=["forward", "pre", "global"])
def test_hooks_run(layer, register):
    model, ran = layer
    seen = []
    handle = register(model.layers_[0].gate_up,
                      lambda t: seen.append(t.shape))
    try:
        _run(model)
    finally:
        handle.remove()
    assert len(seen) == 1 and ran == []
    _run(model)
    assert len(seen) == 1 and ran == ["swiglu"]


def test_replaced_modules_are_called(layer):
    """A wrapper (an adapter, say) around the projection, and a forward set
    on the module itself."""
    model, ran = layer
    block = model.layers_[0]
    plain = block.gate_up

    class Doubled(nn.Module):
        def __init__(self):
            super().__init__()
            self.inner = plain

        def forward(self, x):
            return 2 * self.inner(x)

    before = _run(model)
    ran.clear()
    block.gate_up = Doubled()
    doubled = _run(model)
    assert ran == [] and not torch.allclose(before, doubled)
    block.gate_up = plain
    plain.forward = lambda x: 2 * tp.ColumnParallelLinear.forward(plain, x)
    assert torch.equal(_run(model), doubled) and ran == []
