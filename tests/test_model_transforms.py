"""The model off the GPU's fast paths: on the CPU, under function transforms and
with replaced modules it computes what its modules say, and prepares nothing
that only the HIP kernels read."""

from __future__ import annotations

import pytest
import torch
import torch.nn as nn
from torch.func import functional_call, grad, jvp, vmap

from mini_llm_runtime_amd.model.qwen2 import TinyQwen2Config, TinyQwen2ForCausalLM

IDS = torch.tensor([[1, 7, 3, 9, 2]])  # few enough rows for the fused layer tail


@pytest.fixture
def model():
    torch.manual_seed(0)
    return TinyQwen2ForCausalLM(TinyQwen2Config()).eval()


def _loss(model, params):
    return functional_call(model, params, (IDS,)).square().mean()


def _params(model):
    return {k: p.detach().clone() for k, p in model.named_parameters()}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float64])
def test_cpu_forward_prepares_no_stacked_weight(model, dtype):
    model = model.to(dtype)
    with torch.no_grad():
        model(IDS)
    assert all(layer.mlp._gate_up is None for layer in model.model.layers)


def test_function_transforms(model):
    params = _params(model)
    model(IDS).square().mean().backward()
    got = grad(lambda p: _loss(model, p))(params)
    for name, p in model.named_parameters():
        torch.testing.assert_close(got[name], p.grad)
    # A directional derivative against the gradient it sums over.
    tangents = {k: torch.randn_like(p) for k, p in params.items()}
    _, slope = jvp(lambda p: _loss(model, p), (params,), (tangents,))
    torch.testing.assert_close(slope, sum((got[k] * tangents[k]).sum() for k in params),
                               rtol=1e-4, atol=1e-6)
    stacked = {k: torch.stack([p, p * 1.5]) for k, p in params.items()}
    many = vmap(lambda p: functional_call(model, p, (IDS,)))(stacked)
    for i, factor in enumerate((1.0, 1.5)):
        one = functional_call(model, {k: p * factor for k, p in params.items()}, (IDS,))
        torch.testing.assert_close(many[i], one)


def test_export_and_trace(model):
    with torch.no_grad():
        want = model(IDS)
        torch.testing.assert_close(torch.export.export(model, (IDS,)).module()(IDS), want)
        torch.testing.assert_close(torch.jit.trace(model, (IDS,), check_trace=False)(IDS), want)


class _Wrapped(nn.Module):
    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def forward(self, x):
        return self.inner(x)


@pytest.mark.parametrize("name", ["gate_proj", "up_proj", "down_proj"])
def test_replaced_projections_are_called(model, name):
    with torch.no_grad():
        want = model(IDS)
        for layer in model.model.layers:
            setattr(layer.mlp, name, _Wrapped(getattr(layer.mlp, name)))
        assert torch.equal(model(IDS), want)
