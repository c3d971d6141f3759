"""mlr_rows_linear (kernels/layer_ops.py: linear_silu_mul, apply_linear) against the product in 64 bits.

Bound per output: FP32 sums of k products are off by at most
(k + 2) * 2^-24 * sum |x||w| (any order), and the result is rounded once to
the dtype (half a unit in the last place, relative: 2^-p for p significand
bits, 2^-8 bf16, 2^-11 fp16, 2^-24 FP32). The gated form is compared with silu_mul over the two products,
each within that bound: silu is 1.1-Lipschitz and each of its two roundings
adds one more half unit.
"""

from __future__ import annotations

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from mini_llm_runtime_amd import _lib
from mini_llm_runtime_amd.kernels import layer_ops as kops

pytestmark = pytest.mark.gpu

HALF_ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}
DTYPES = list(HALF_ULP)
# Row tiles (16, 32) and their edges, ragged columns, k below one block, not a
# whole number of blocks, several load batches, and long enough to be split.
SHAPES = [(1, 16, 8), (2, 17, 72), (15, 40, 136), (16, 1152, 896), (3, 896, 4864), (16, 100, 8200),
          (17, 33, 64), (32, 896, 4864), (31, 50, 1000)]


def _inputs(rows, n, k, dtype, device):
    gen = torch.Generator().manual_seed(rows * 7 + n + k)
    x = torch.randn(rows, k, generator=gen).to(dtype).to(device)
    w = (torch.randn(n, k, generator=gen) * k ** -0.5).to(dtype).to(device)
    b = torch.randn(n, generator=gen).to(dtype).to(device)
    return x, w, b


def _bound(x, w, y, dtype):
    mass = x.double().abs() @ w.double().abs().t() + y.abs()
    return HALF_ULP[dtype] * y.abs() * 1.01 + (x.shape[1] + 2) * 2.0 ** -24 * mass + 2.0 ** -25


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d)[6:])
@pytest.mark.parametrize("rows,n,k", SHAPES)
def test_rows_linear_matches_float64(device, dtype, rows, n, k):
    x, w, b = _inputs(rows, n, k, dtype, device)
    took = kops._rows_linear(x, w, b, False)
    if rows > 16 and dtype is torch.float32:
        assert took is None  # the library's
        return
    for bias in (b, None):
        got = kops._rows_linear(x, w, bias, False)
        want = F.linear(x.double(), w.double(), None if bias is None else bias.double())
        assert bool(((got.double() - want).abs() <= _bound(x, w, want, dtype)).all())
    # Strided rows and a leading dimension give the same bits.
    wide = torch.zeros(rows, k + 64, dtype=dtype, device=device)
    wide[:, :k] = x
    assert torch.equal(kops._rows_linear(wide[:, :k], w, b, False), took)
    assert torch.equal(kops._rows_linear(x[:, None], w, b, False), took[:, None])
    if rows <= 16:  # a row does not depend on its neighbours
        assert torch.equal(kops._rows_linear(x[:1], w, b, False), took[:1])


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d)[6:])
@pytest.mark.parametrize("rows,n,k", [(1, 16, 8), (16, 40, 136), (16, 4864, 896), (32, 33, 1000)])
def test_gated_form_matches_the_two_products(device, dtype, rows, n, k):
    x, w, _ = _inputs(rows, 2 * n, k, dtype, device)
    got = kops.linear_silu_mul(x, w).double()
    y = F.linear(x.double(), w.double())
    off = _bound(x, w, y, dtype)
    g, u, dg, du = y[:, :n], y[:, n:], off[:, :n], off[:, n:]
    s = F.silu(g)
    h = HALF_ULP[dtype] + 2.0 ** -22
    ds = 1.1 * dg + h * (s.abs() + 1.1 * dg) + 2.0 ** -25
    want = s * u
    bound = (s.abs() + ds) * du + ds * u.abs()
    bound = bound + h * (want.abs() + bound) + 2.0 ** -25
    assert bool(((got - want).abs() <= bound).all())


def test_calls_that_stay_with_torch(device):
    """Hooks, gradients, autocast, subclasses and operands the kernel does not
    read give what the module gives."""
    layer = nn.Linear(64, 32, device=device, dtype=torch.bfloat16)
    x = torch.randn(4, 64, device=device, dtype=torch.bfloat16)
    assert kops.apply_linear(layer, x).grad_fn is not None
    with torch.no_grad():
        seen = []
        handle = layer.register_forward_hook(lambda m, i, o: seen.append(o))
        kops.apply_linear(layer, x)
        assert len(seen) == 1
        handle.remove()
        with torch.autocast("cuda", dtype=torch.float16):
            assert kops.apply_linear(layer, x).dtype == layer(x).dtype
        for odd in (x.t().contiguous().t(), x[:1].expand(4, 64), x[:0]):
            assert torch.allclose(kops.apply_linear(layer, odd).float(), layer(odd).float(),
                                  atol=2e-2)
        assert kops._rows_linear(x.t().contiguous().t(), layer.weight, None, False) is None
        assert kops._rows_linear(x[:1].expand(4, 64), layer.weight, None, False) is None
        odd = torch.randn(4, 65, device=device, dtype=torch.bfloat16)[:, 1:]
        assert kops._rows_linear(odd, layer.weight, None, False) is None
        with pytest.raises(RuntimeError):
            kops.apply_linear(layer, x[:, :32])


def test_entry_point_refuses_what_the_kernel_cannot_take(device):
    lib = _lib.load()
    x = torch.zeros(33, 64, device=device, dtype=torch.bfloat16)
    w = torch.zeros(32, 64, device=device, dtype=torch.bfloat16)
    out = torch.full((33, 32), 3.0, device=device, dtype=torch.bfloat16)

    def call(rows=4, xs=64, k=64, xp=x.data_ptr(), dtype=2, n=32, nbytes=0):
        return lib.mlr_rows_linear(xp, xs, w.data_ptr(), None, out.data_ptr(), 32, rows, n, k, 0,
                                   dtype, None, nbytes, _lib.stream_handle(device))

    assert call(rows=33) != 0 and call(xs=63) != 0 and call(xp=x.data_ptr() + 2) != 0
    assert call(dtype=3) != 0 and call(k=0) != 0 and call(n=0) != 0
    assert call(k=8192, xs=8192) == 3  # split over workgroups: needs its workspace
    torch.cuda.synchronize()
    assert bool((out == 3.0).all())
