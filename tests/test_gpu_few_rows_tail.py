"""The fused tail of a decoder layer over a decode step's few rows
(mlr_norm_rows_linear, mlr_rms_norm_sums) against the separate calls: the
residual, the norms and the down projection bit for bit; the gated products
too where both calls deal their k blocks to the same waves, elsewhere within
FP32 sums in another order."""

from __future__ import annotations

import pytest
import torch
import torch.nn as nn

from mini_llm_runtime_amd import _lib
from mini_llm_runtime_amd.kernels import layer_ops as kops
from mini_llm_runtime_amd.model.qwen2 import Qwen2DecoderLayer, TinyQwen2Config

pytestmark = pytest.mark.gpu
HALF = [torch.bfloat16, torch.float16]


def _rand(gen, *shape, dtype, device, scale=1.0):
    return (torch.randn(*shape, generator=gen) * scale).to(dtype).to(device)


@pytest.mark.parametrize("dtype", HALF, ids=lambda t: str(t)[6:])
@pytest.mark.parametrize("rows,k,n", [(1, 8, 16), (3, 64, 128), (16, 896, 4864), (15, 1024, 33),
                                      (17, 896, 300), (32, 1008, 48), (5, 520, 17)])
def test_norm_and_gated_product_match_the_two_calls(device, dtype, rows, k, n):
    gen = torch.Generator().manual_seed(rows + k)
    x, res = (_rand(gen, rows, 1, k, dtype=dtype, device=device, scale=2) for _ in range(2))
    nw = _rand(gen, k, dtype=dtype, device=device)
    w = _rand(gen, 2 * n, k, dtype=dtype, device=device, scale=k ** -0.5)
    got, res_out = kops.norm_silu_mul(x, res, nw, 1e-6, w)
    normed, want_res = kops.rms_norm(x, nw, 1e-6, residual=res)
    assert torch.equal(res_out, want_res)
    want = kops.linear_silu_mul(normed, w)
    # Same k blocks, but dealt to other wave counts at some sizes: FP32 sums in
    # another order move a result by one rounding at most now and then.
    ulp = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype]
    off = (got.double() - want.double()).abs()
    assert bool((off <= 4 * ulp * want.double().abs() + 1e-4).all())
    if k == 896 and rows <= 16:
        assert torch.equal(got, want)
    wide = torch.zeros(rows, 1, k + 64, dtype=dtype, device=device)
    wide[..., :k] = x
    again, _ = kops.norm_silu_mul(wide[..., :k], res, nw, 1e-6, w)
    assert torch.equal(again, got)


@pytest.mark.parametrize("dtype", HALF + [torch.float32], ids=lambda t: str(t)[6:])
@pytest.mark.parametrize("rows,n", [(1, 896), (16, 896), (3, 64), (9, 1024), (2, 1000)])
def test_norm_of_a_products_parts(device, dtype, rows, n):
    k = 8448 if dtype is not torch.float32 else 4224
    gen = torch.Generator().manual_seed(n)
    x = _rand(gen, rows, 1, k, dtype=dtype, device=device)
    w = _rand(gen, n, k, dtype=dtype, device=device, scale=k ** -0.5)
    res = _rand(gen, rows, 1, n, dtype=dtype, device=device)
    nw = _rand(gen, n, dtype=dtype, device=device)
    parts = kops._rows_linear(x, w, None, False, sums=True)
    assert isinstance(parts, kops.RowSums) and parts.shape == (rows, 1, n)
    whole = kops._rows_linear(x, w, None, False)
    assert torch.equal(parts.tensor(), whole)
    got = kops.rms_norm_sums(parts, nw, 1e-6, res)
    want = kops.rms_norm(whole, nw, 1e-6, residual=res)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("dtype", HALF + [torch.float32], ids=lambda t: str(t)[6:])
@pytest.mark.parametrize("rows", [1, 16, 32, 33])
def test_layer_tail_matches_the_modules(device, monkeypatch, dtype, rows):
    config = TinyQwen2Config(hidden_size=896, intermediate_size=4864, num_attention_heads=14,
                             num_key_value_heads=2)
    torch.manual_seed(0)
    with device:
        layer = Qwen2DecoderLayer(config).to(dtype).eval()
    x = torch.randn(rows, 1, 896, device=device).to(dtype)
    with torch.no_grad():
        took = layer._few_rows_tail(x, x)
        assert (took is not None) == (rows <= 32 and dtype is not torch.float32)
        got = layer._block(x, lambda h: h * 0.5)
        residual, delta = layer._block_parts(x, None, lambda h: h * 0.5)
        nxt = layer.input_layernorm.forward_with_residual(delta, residual)
        monkeypatch.setattr(Qwen2DecoderLayer, "_few_rows_tail", lambda *a: None)
        want = layer._block(x, lambda h: h * 0.5)
        residual, delta = layer._block_parts(x, None, lambda h: h * 0.5)
        same = layer.input_layernorm.forward_with_residual(delta, residual)
    if rows <= 16 or rows == 33 or dtype is torch.float32:
        assert torch.equal(got, want)
        assert torch.equal(nxt[0], same[0]) and torch.equal(nxt[1], same[1])
    else:  # 32 rows: other wave counts, see above
        assert ((got - want).float().norm() / want.float().norm()).item() < 2e-2


def test_tail_leaves_hooks_and_gradients_alone(device):
    layer = Qwen2DecoderLayer(TinyQwen2Config()).to(device, torch.bfloat16).eval()
    x = torch.randn(4, 1, 64, device=device, dtype=torch.bfloat16)
    assert layer._few_rows_tail(x, x) is None  # the norm's weight wants a gradient
    with torch.no_grad():
        assert layer._few_rows_tail(x, x) is not None
        for module in (layer.mlp, layer.post_attention_layernorm, layer.mlp.down_proj):
            handle = module.register_forward_hook(lambda *a: None)
            assert layer._few_rows_tail(x, x) is None
            handle.remove()
        layer.mlp.down_proj = nn.Sequential(layer.mlp.down_proj)
        assert layer._few_rows_tail(x, x) is None


def test_biased_down_projection(device):
    """A down projection with a bias whose k is split over workgroups: the tail
    sums it, with the bits of the module's own product."""
    config = TinyQwen2Config(hidden_size=896, intermediate_size=4864, num_attention_heads=14,
                             num_key_value_heads=2)
    torch.manual_seed(0)
    layer = Qwen2DecoderLayer(config)
    layer.mlp.down_proj = nn.Linear(4864, 896)
    layer = layer.to(device, torch.bfloat16).eval()
    x = torch.randn(4, 1, 896, device=device, dtype=torch.bfloat16)
    with torch.no_grad():
        residual, delta = layer._few_rows_tail(x, x)
        gated, same = kops.norm_silu_mul(x, x, layer.post_attention_layernorm.weight, 1e-6,
                                         layer.mlp._gate_up_weight())
        want = torch.nn.functional.linear(gated.double(), layer.mlp.down_proj.weight.double(),
                                          layer.mlp.down_proj.bias.double())
    assert torch.equal(residual, same)
    # One rounding to bf16, and FP32 sums of 4,864 products.
    assert ((delta.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all()


def test_entry_points_refuse(device):
    lib = _lib.load()
    b = torch.zeros(64, 1024, device=device, dtype=torch.bfloat16)
    o = torch.zeros_like(b)
    s = _lib.stream_handle(device)

    def call(rows=4, k=64, xs=64, out_res=o.data_ptr(), xp=b.data_ptr(), dtype=2):
        return lib.mlr_norm_rows_linear(xp, xs, b.data_ptr(), 64, out_res, b.data_ptr(), 1e-6,
                                        b.data_ptr(), o.data_ptr(), 16, rows, 16, k, dtype, s)

    assert call(rows=33) and call(k=12) and call(k=1032, xs=1032) and call(xs=60)
    assert call(out_res=b.data_ptr()) and call(xp=b.data_ptr() + 2) and call(dtype=0)
    assert call(rows=17, k=1016, xs=1016)
    f = torch.zeros(1024, device=device)
    for hidden, splits in ((12, 1), (4096, 1), (64, 0), (64, 65)):
        assert lib.mlr_rms_norm_sums(f.data_ptr(), splits, b.data_ptr(), hidden, o.data_ptr(),
                                     b.data_ptr(), o.data_ptr(), 1, hidden, 1e-6, 2, s)
