"""The whole-prompt prefill's fused rotation and cache write
(mlr_qkv_rope_write_prompt) against the PyTorch rotation and write_slots it
replaces: the same bits, in the layer's output, the cache and the fresh rows."""

from __future__ import annotations

import pytest
import torch

from mini_llm_runtime_amd.kernels import pre_attention as kpre
from mini_llm_runtime_amd.model.qwen2 import TinyQwen2Config
from mini_llm_runtime_amd.model.qwen2_attention import Qwen2Attention
from mini_llm_runtime_amd.runtime.paged_kv_cache import PagedKVCache

pytestmark = pytest.mark.gpu


def _layer(hidden, hq, hkv, dtype, device, seed=0):
    torch.manual_seed(seed)
    config = TinyQwen2Config(hidden_size=hidden, intermediate_size=64, num_attention_heads=hq,
                             num_key_value_heads=hkv)
    return Qwen2Attention(config).to(device=device, dtype=dtype).eval()


def _run(layer, x, pos, slots, dtype, device, blocks, block_size, layer_idx=1):
    cache = PagedKVCache(2, blocks, block_size, layer.num_key_value_heads, layer.head_dim,
                         dtype=dtype, device=device)
    cache.k_cache.fill_(0.5)
    cache.v_cache.fill_(-0.5)
    with torch.no_grad():
        out = layer.forward_prefill_with_cache(x, pos, cache, layer_idx, slots)
    return out, cache.k_cache, cache.v_cache


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16],
                         ids=lambda t: str(t)[6:])
@pytest.mark.parametrize("hidden,hq,hkv,tokens", [
    (64, 4, 2, 1), (64, 4, 2, 37), (896, 14, 2, 1021), (1536, 12, 2, 130), (60, 6, 3, 20),
    (80, 1, 1, 33), (320, 2, 1, 50)])
def test_fused_prompt_equals_unfused(device, monkeypatch, dtype, hidden, hq, hkv, tokens):
    layer = _layer(hidden, hq, hkv, dtype, device)
    gen = torch.Generator().manual_seed(tokens)
    x = torch.randn(1, tokens, hidden, generator=gen).to(dtype).to(device)
    blocks = tokens // 4 + 9
    slots = torch.randperm(blocks * 4, generator=gen)[:tokens].to(device)
    for pos_dtype, slot_dtype in ((torch.int64, torch.int64), (torch.int32, torch.int32)):
        pos = (torch.arange(tokens) * 3 + 70000)[None].to(device, pos_dtype)
        args = (layer, x, pos, slots.to(slot_dtype), dtype, device, blocks, 4)
        assert layer._prompt_fusable(x, pos, PagedKVCache(2, 1, 4, hkv, hidden // hq, dtype=dtype,
                                                          device=device), 1, slots)
        got = _run(*args)
        with monkeypatch.context() as m:
            m.setattr(Qwen2Attention, "_prompt_fusable", lambda *a: False)
            want = _run(*args)
        for g, w in zip(got, want):
            assert torch.equal(g, w)


def test_strided_projections_and_skipped_slots(device):
    """Slices of one wide buffer as q, k and v; a slot outside the pool is not
    written, its fresh row is."""
    d, hq, hkv, tokens = 64, 4, 2, 21
    cache = PagedKVCache(1, 4, 16, hkv, d, dtype=torch.bfloat16, device=device)
    cache.k_cache.zero_()
    cache.v_cache.zero_()
    wide = torch.randn(tokens, (hq + 2 * hkv) * d, device=device).bfloat16()
    q, k, v = (wide[:, a * d:b * d].view(tokens, b - a, d)
               for a, b in ((0, hq), (hq, hq + hkv), (hq + hkv, hq + 2 * hkv)))
    freq = 1.0 / 10000 ** (torch.arange(0, d, 2, device=device) / d)
    pos = torch.arange(tokens, device=device)
    slots = torch.arange(tokens, device=device) + 40
    slots[5] = 64
    out, fk, fv = kpre.qkv_rope_write_prompt(q, k, v, pos, freq, cache, 0, slots, 32)
    same = kpre.qkv_rope_write_prompt(q.contiguous(), k.contiguous(), v.contiguous(), pos, freq,
                                      cache, 0, slots, 32)
    want = kpre.qkv_rope_write(wide, pos, freq, cache, 0, torch.arange(tokens, device=device), hq)
    assert torch.equal(out, want) and torch.equal(same[0], want)
    rows_k, rows_v = (c[0].reshape(-1, hkv, d) for c in (cache.k_cache, cache.v_cache))
    assert torch.equal(fk[:tokens], rows_k[:tokens]) and torch.equal(fv[:tokens], rows_v[:tokens])
    kept = [i for i in range(tokens) if i != 5]
    assert torch.equal(rows_k[slots[kept]], fk[:tokens][kept])
    assert not rows_k[45].any() and not rows_v[45].any()


def test_what_keeps_the_torch_rotation(device):
    layer = _layer(64, 4, 2, torch.float32, device)
    x = torch.randn(1, 5, 64, device=device)
    pos = torch.arange(5, device=device)[None]
    slots = torch.arange(5, device=device)
    seen = []
    handle = layer.rotary_embedding.register_forward_hook(lambda *a: seen.append(1))
    _run(layer, x, pos, slots, torch.float32, device, 2, 16)
    handle.remove()
    assert seen == [1]
    _run(layer, x, pos, slots, torch.bfloat16, device, 2, 16)  # the cache converts
    _run(layer, x, pos.float(), slots, torch.float32, device, 2, 16)
    cache = PagedKVCache(2, 2, 16, 2, 16, dtype=torch.float32, device=device)
    for bad, error in ((slots + 30, IndexError), (slots * 0, ValueError)):
        with pytest.raises(error):
            layer.forward_prefill_with_cache(x, pos, cache, 0, bad)
    with pytest.raises(IndexError, match="layer_idx"):
        layer.forward_prefill_with_cache(x, pos, cache, 2, slots)


def test_replaced_projection_without_weights(device):
    """A projection module without q_proj is called, as for any other path."""
    class Wrapped(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def forward(self, x):
            return self.inner(x)

    layer = _layer(64, 4, 2, torch.bfloat16, device)
    x = torch.randn(1, 5, 64, device=device).bfloat16()
    pos, slots = torch.arange(5, device=device)[None], torch.arange(5, device=device)
    want = _run(layer, x, pos, slots, torch.bfloat16, device, 2, 16)
    layer.qkv_proj = Wrapped(layer.qkv_proj)
    for g, w in zip(_run(layer, x, pos, slots, torch.bfloat16, device, 2, 16), want):
        assert torch.equal(g, w)
