"""The dense MLP against its layers called one by one."""

import pytest
import torch

import fusioninfer_amd.ops as ops
from fusioninfer_amd.models.model import MLP
from fusioninfer_amd.models.registry import get_model_config


@pytest.fixture
def mlp():
    m = MLP(get_model_config("tiny-qwen3"))
    g = torch.Generator().manual_seed(1)
    for p in m.parameters():
        p.data.normal_(0, 0.1, generator=g)
    return m


def _x(mlp):
    w = mlp.gate_up_proj.weight
    return torch.randn(3, w.shape[1], generator=torch.Generator()
                       .manual_seed(2)).to(w.dtype)


def _one_by_one(mlp, x):
    return mlp.down_proj(ops.silu_and_mul(mlp.gate_up_proj(x)))


def test_mlp_is_its_layers(mlp):
    x = _x(mlp)
    assert torch.equal(mlp(x), _one_by_one(mlp, x))


@pytest.mark.parametrize("hook", ["forward", "pre", "global"])
def test_mlp_calls_the_hooks_of_gate_up(mlp, hook):
    x, seen = _x(mlp), []

    def forward(module, args, out):
        if module is mlp.gate_up_proj:
            seen.append(out.shape)
            return out * 2

    def pre(module, args):
        seen.append(args[0].shape)
        return (args[0] * 2,)

    plain = mlp(x)
    handle = {
        "forward": lambda: mlp.gate_up_proj.register_forward_hook(forward),
        "pre": lambda: mlp.gate_up_proj.register_forward_pre_hook(pre),
        "global": lambda: torch.nn.modules.module.
        register_module_forward_hook(forward),
    }[hook]()
    try:
        got, want = mlp(x), _one_by_one(mlp, x)
    finally:
        handle.remove()
    assert len(seen) == 2 and torch.equal(got, want)
    assert not torch.equal(got, plain)


def test_mlp_takes_a_bias_another_forward_or_another_module(mlp):
    x = _x(mlp)
    layer = mlp.gate_up_proj
    layer.bias = torch.nn.Parameter(torch.ones_like(layer.weight[:, 0]))
    assert torch.equal(mlp(x), _one_by_one(mlp, x))
    layer.bias = None
    layer.forward = lambda v: torch.nn.functional.linear(v, layer.weight) + 1
    assert torch.equal(mlp(x), _one_by_one(mlp, x))
    del layer.forward

    class Halved(torch.nn.Module):
        def forward(self, v):
            return layer(v) / 2

    mlp.gate_up_proj = Halved()
    assert torch.equal(mlp(x), _one_by_one(mlp, x))
