"""A step's prefills and decodes in one pass over the layers against the two
forwards run one after the other.

The two differ only in the row count of the library GEMMs (which may pick
another kernel, i.e. another order of FP32 sums): FP32 logits within 1e-4
relative, 16-bit logits within the rounding that a layer's output carries on
(relative 2-norm 2e-2). Cache rows outside the step's slots keep their bits."""

from __future__ import annotations

import contextlib

import pytest
import torch

from mini_llm_runtime_amd.kernels import paged_attention as kpa
from mini_llm_runtime_amd.model.qwen2 import TinyQwen2Config, TinyQwen2ForCausalLM
from mini_llm_runtime_amd.runtime import model_runner
from mini_llm_runtime_amd.runtime.paged_kv_cache import PagedKVCache
from mini_llm_runtime_amd.runtime.request import RequestStatus

pytestmark = pytest.mark.gpu
P, D = RequestStatus.PREFILLING, RequestStatus.DECODING


def _setup(config, dtype, device, order, block_size):
    """order: (phase, context, tokens) per request."""
    torch.manual_seed(1)
    with device:
        model = TinyQwen2ForCausalLM(config).to(dtype).eval()
    gen = torch.Generator().manual_seed(len(order))
    need = [-(-n // block_size) for _, n, _ in order]
    perm = torch.randperm(sum(need) + 2, generator=gen).tolist()
    caches = []
    for _ in range(2):
        cache = PagedKVCache(config.num_hidden_layers, sum(need) + 2, block_size,
                             config.num_key_value_heads, config.head_dim, dtype=dtype,
                             device=device)
        for c in (cache.k_cache, cache.v_cache):
            c.copy_(torch.randn(c.shape, generator=torch.Generator().manual_seed(5)).to(dtype))
        caches.append(cache)
    tables, pos, slots, qsl = [], [], [], [0]
    for i, (_, n, count) in enumerate(order):
        tables.append(perm[sum(need[:i]):sum(need[:i + 1])])
        pos += range(n - count, n)
        slots += [tables[-1][p // block_size] * block_size + p % block_size
                  for p in range(n - count, n)]
        qsl.append(qsl[-1] + count)
    t = lambda v: torch.tensor(v, dtype=torch.long, device=device)  # noqa: E731
    width = max(need)
    batch = model_runner.ModelBatch(
        [f"r{i}" for i in range(len(order))],
        torch.randint(0, config.vocab_size, (qsl[-1],), generator=gen).to(device), t(pos), t(qsl),
        [phase for phase, _, _ in order], t([n for _, n, _ in order]),
        t([x + [-1] * (width - len(x)) for x in tables]), t(slots))
    return model, batch, caches


SMALL = TinyQwen2Config()
WIDE = TinyQwen2Config(vocab_size=515, hidden_size=896, intermediate_size=300, num_hidden_layers=2,
                       num_attention_heads=14, num_key_value_heads=2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16],
                         ids=lambda t: str(t)[6:])
@pytest.mark.parametrize("config,block_size,order", [
    (SMALL, 16, [(P, 5, 5), (D, 9, 1)]),
    (SMALL, 4, [(D, 1, 1), (P, 30, 30), (D, 33, 1), (P, 20, 7)]),
    (WIDE, 16, [(P, 300, 300), (P, 90, 40), (D, 700, 1), (D, 16, 1), (D, 17, 1)]),
    (WIDE, 16, [(P, 300, 300), (D, 200, 1), (P, 1, 1), (D, 33, 1)])])
def test_mixed_step_equals_the_two_forwards(device, monkeypatch, dtype, config, block_size, order):
    model, batch, caches = _setup(config, dtype, device, order, block_size)
    assert model_runner._takes_mixed_steps(model, device)
    with torch.no_grad():
        got = model_runner.execute_model_batch(model, batch, caches[0])
        monkeypatch.setattr(model_runner, "_takes_mixed_steps", lambda *a: False)
        want = model_runner.execute_model_batch(model, batch, caches[1])
    tol = 1e-4 if dtype is torch.float32 else 2e-2
    assert ((got - want).double().norm() / want.double().norm()).item() <= tol
    slots = batch.slot_mapping.tolist()
    kept = torch.ones(caches[0].num_blocks * block_size, dtype=torch.bool)
    kept[slots] = False
    for a, b in ((caches[0].k_cache, caches[1].k_cache), (caches[0].v_cache, caches[1].v_cache)):
        a, b = (c.flatten(1, 2).cpu().double() for c in (a, b))
        assert torch.equal(a[:, kept], b[:, kept])
        assert ((a - b).norm() / b[:, slots].norm()).item() <= tol


def test_steps_that_keep_the_two_forwards(device):
    model, batch, caches = _setup(SMALL, torch.float32, device, [(P, 5, 5), (D, 9, 1)], 16)
    seen = []
    handle = model.model.layers[1].mlp.register_forward_hook(lambda m, i, o: seen.append(o.shape))
    with torch.no_grad():
        model_runner.execute_model_batch(model, batch, caches[0])
        assert len(seen) == 2
        handle.remove()
        layer = model.model.layers[0]
        layer.self_attn.forward_decode_batch_with_cache = (
            lambda *a, **k: seen.append(1) or type(layer.self_attn).forward_decode_batch_with_cache(
                layer.self_attn, *a, **k))
        model_runner.execute_model_batch(model, batch, caches[1])
        assert seen[2:] == [1]


@pytest.mark.parametrize("mixed", [True, False])
def test_under_a_default_device(device, monkeypatch, mixed):
    """A step, a slot write and a checked decode inside a torch.device context,
    where tensors made without a device land on the GPU."""
    model, batch, caches = _setup(SMALL, torch.float32, device, [(P, 5, 5), (D, 9, 1)], 16)
    if not mixed:
        monkeypatch.setattr(model_runner, "_takes_mixed_steps", lambda *a: False)
    rows = torch.ones(2, 2, 16, device=device)
    slots = torch.tensor([3, 40], device=device)
    q = torch.ones(2, 4, 16, device=device)
    args = (batch.block_tables, batch.context_lens, 16)
    results = []
    for cache, context in zip(caches, (torch.device("cuda"), contextlib.nullcontext())):
        with torch.no_grad(), context:
            logits = model_runner.execute_model_batch(model, batch, cache)
            cache.write_slots(slot_mapping=slots, k=rows, v=rows, layer_idx=0)
            k, v = cache.get_layer_cache(0)
            results.append((logits, k, kpa.paged_attention_decode_batch_parallel(q, k, v, *args)))
    for got, want in zip(*results):
        assert (got - want).norm() <= 1e-4 * want.norm()


def test_hooks_on_norms_see_the_two_forwards(device):
    """The first layer's input norm is called as a module, once per forward."""
    model, batch, caches = _setup(SMALL, torch.float32, device, [(P, 5, 5), (D, 9, 1)], 16)
    seen = []
    norm = model.model.layers[0].input_layernorm
    handle = norm.register_forward_hook(lambda m, i, o: seen.append(o.numel() // 64))
    with torch.no_grad():
        model_runner.execute_model_batch(model, batch, caches[0])
        handle.remove()
        assert seen == [5, 1]
        last = model.model.norm
        add = last.forward_with_residual
        last.forward_with_residual = lambda x, r: seen.append(r.numel() // 64) or add(x, r)
        model_runner.execute_model_batch(model, batch, caches[1])
    assert seen[2:] == [5, 1]
