"""RMSNorm (with the residual add before it), the MLP's silu(gate) * up and
linear layers over a decode step's few rows on the HIP library: one launch each
where PyTorch issues several.

``rms_norm`` computes what ``Qwen2RMSNorm.forward`` computes (reference
model/qwen2.py:88-123) and ``silu_mul`` what ``F.silu(gate) * up`` in
``Qwen2MLP.forward`` (:768-792) computes, with the same roundings (see
csrc/layer_ops.hip); the decoder layer's residual add before its
post-attention norm rides on ``rms_norm(..., residual=...)``. bf16, fp16 and
FP32 on a HIP device; there is no PyTorch fallback. ``apply_linear``,
``linear_silu_mul``, ``norm_silu_mul`` and ``rms_norm_sums`` stream the weights
of a linear layer once for a few rows (up to 32 in 16 bits, 16 in FP32;
csrc/rows_linear.hip), with the norm before it (16 bits) or the activation
after it in the same launch; more rows go to the library's GEMM.
"""

from __future__ import annotations

import torch
import torch.nn as nn
import torch.nn.functional as F

from .. import _lib

DTYPES = (torch.bfloat16, torch.float16, torch.float32)


def supported(x: torch.Tensor) -> bool:
    """Whether these kernels take `x` (a HIP tensor of a supported dtype)."""
    return x.is_cuda and x.dtype in DTYPES


def _rows(t: torch.Tensor, name: str) -> torch.Tensor:
    """`t` as [rows, last] with unit stride along the last dimension."""
    if t.stride(-1) != 1:
        t = t.contiguous()
    rows = t.reshape(-1, t.shape[-1])
    if rows.numel() and rows.stride(-1) != 1:
        raise ValueError(f"{name} must be unit-stride along its last dimension")
    return rows


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float,
             residual: torch.Tensor | None = None):
    """weight * x / sqrt(mean(x^2) + eps) over the last dimension.

    With `residual`: r = residual + x (rounded to the dtype) is normalised
    instead, and (normalised, r) is returned; r is a new tensor."""
    if not supported(x):
        raise ValueError("rms_norm needs a bf16, fp16 or fp32 tensor on a HIP device")
    hidden = x.shape[-1]
    if weight.shape != (hidden,) or weight.dtype != x.dtype or weight.device != x.device:
        raise ValueError("weight must have shape [hidden] and x's dtype and device")
    if residual is not None and (residual.shape != x.shape or residual.dtype != x.dtype
                                 or residual.device != x.device):
        raise ValueError("residual must match x in shape, dtype and device")
    xr = _rows(x, "x")
    weight = weight.contiguous()
    out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
    rows = xr.shape[0]
    xs = xr.stride(0) if rows else hidden
    rp = rs = res_out = ro = None
    if residual is not None:
        rr = _rows(residual, "residual")
        rp, rs = rr.data_ptr(), rr.stride(0) if rows else hidden
        res_out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        ro = res_out.data_ptr()
    device = x.device
    with _lib.on(device):
        status = _lib.load().mlr_rms_norm(
            xr.data_ptr(), xs, rp, hidden if rs is None else rs, ro, hidden, weight.data_ptr(),
            out.data_ptr(), hidden, rows, hidden, float(eps), _lib.DTYPE_CODES[x.dtype],
            _lib.stream_handle(device))
    _lib.check(status, "mlr_rms_norm")
    return out if residual is None else (out, res_out)


def silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    """silu(gate) * up for gate_up = [..., 2 * intermediate] (the gate in the
    first half of the last dimension, up in the second)."""
    if not supported(gate_up):
        raise ValueError("silu_mul needs a bf16, fp16 or fp32 tensor on a HIP device")
    if gate_up.shape[-1] % 2:
        raise ValueError("gate_up's last dimension must be 2 * intermediate")
    inter = gate_up.shape[-1] // 2
    g = _rows(gate_up, "gate_up")
    out = torch.empty(*gate_up.shape[:-1], inter, dtype=gate_up.dtype, device=gate_up.device)
    rows = g.shape[0]
    lib = _lib.load()
    with _lib.on(gate_up.device):
        status = lib.mlr_silu_mul(g.data_ptr(), g.stride(0) if rows else 2 * inter,
                                  out.data_ptr(), inter, rows, inter,
                                  _lib.dtype_code(gate_up.dtype, "silu_mul"),
                                  _lib.stream_handle(gate_up.device))
    _lib.check(status, "mlr_silu_mul")
    return out


# ---------------------------------------------------------------------------
# Linear layers over a decode step's few rows
# ---------------------------------------------------------------------------
_MB = 1 << 20
# Largest weight, in bytes, that mlr_rows_linear takes by (16-bit, rows above
# 16, gated): a few rows make the product a read of the weight, and the GEMM
# library is as good at that once the weight fills its tiles. Measured in
# graphs on cold weights, us, kernel / library (gated: library GEMM + silu_mul):
# bf16, 16 rows: 896x4864 7.7 / 17.1, 3584x3584 10.4 / 12.1, 4608x3584
# 16.5 / 12.3; gated 896x4864 8.4 / 11.3, 1536x8960 16.7 / 42.0, 3584x18944
# 65 / 61. 32 rows: 896x4864 9.6 / 13.3, 2048x2048 9.7 / 11.3, 3584x3584
# 15.1 / 11.9; gated 896x4864 11.2 / 14.3, 2048x5632 22.2 / 19.2. FP32, 16
# rows: 4864x896 10.3 / 15.1, 3584x3584 18.6 / 14.1; gated 896x4864
# 13.5 / 15.2, 2048x5632 27.5 / 25.0; at 32 rows the library wins.
_ROWS_LIMIT = {
    (True, False, False): 28 * _MB, (True, False, True): 64 * _MB,
    (True, True, False): 16 * _MB, (True, True, True): 20 * _MB,
    (False, False, False): 28 * _MB, (False, False, True): 40 * _MB,
    (False, True, False): 0, (False, True, True): 0,
}


def _transformed() -> bool:
    """Whether something is to see the call as torch operations: tracing,
    compilation, a dispatch or function mode, a functorch transform, forward
    differentiation or autocast."""
    c = torch._C
    return (torch.is_autocast_enabled() or c._get_tracing_state() is not None
            or c._len_torch_dispatch_stack() > 0 or c._len_torch_function_stack() > 0
            or c._functorch.peek_interpreter_stack() is not None
            or torch.autograd.forward_ad._current_level >= 0
            or torch.compiler.is_compiling())


def _rows_linear(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None,
                 gated: bool, sums: bool = False) -> torch.Tensor | RowSums | None:
    """The product by mlr_rows_linear, or None for a call that it does not
    take (the caller then runs the PyTorch operations). With ``sums`` a product
    whose k is split over workgroups comes back as its parts."""
    dtype = x.dtype
    if not x.is_cuda or weight.dtype != dtype or dtype not in DTYPES or weight.ndim != 2:
        return None
    if torch._C._get_tracing_state() is not None:  # sizes would be tensors
        return None
    n, k = weight.shape
    if x.ndim < 2 or x.shape[-1] != k or k == 0:
        return None
    rows, size = x.numel() // k, dtype.itemsize
    if (rows == 0 or rows > 32
            or n * k * size > _ROWS_LIMIT[size == 2, rows > 16, gated]):
        return None
    if (weight.device != x.device or not weight.is_contiguous() or k * size % 16
            or x.stride(-1) != 1 or type(x) is not torch.Tensor
            or type(weight) not in (torch.Tensor, nn.Parameter)):
        return None
    if bias is not None and (bias.dtype != dtype or bias.device != x.device
                             or bias.shape != (n,) or not bias.is_contiguous()
                             or type(bias) not in (torch.Tensor, nn.Parameter)):
        return None
    if torch.is_grad_enabled() and (x.requires_grad or weight.requires_grad
                                    or (bias is not None and bias.requires_grad)):
        return None
    xr = x.reshape(rows, k)
    stride = xr.stride(0) if rows > 1 else k
    if stride < k or stride >= 1 << 22 or stride * size % 16 or xr.stride(1) != 1:
        return None
    xp, wp = xr.data_ptr(), weight.data_ptr()
    if (xp | wp) & 15 or _transformed():
        return None
    n_out = n // 2 if gated else n
    device = x.device
    lib = _lib.load()
    code = _lib.DTYPE_CODES[dtype]
    nbytes = lib.mlr_rows_linear_workspace_size(rows, n_out, k, gated, code)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=device) if nbytes else None
    out = None
    if not (sums and nbytes):
        sums = False
        out = torch.empty((*x.shape[:-1], n_out), dtype=dtype, device=device)
    with _lib.on(device):
        status = lib.mlr_rows_linear(
            xp, stride, wp, bias.data_ptr() if bias is not None else None,
            out.data_ptr() if out is not None else None, n_out,
            rows, n_out, k, gated, code, ws.data_ptr() if ws is not None else None, nbytes,
            _lib.stream_handle(device))
    _lib.check(status, "mlr_rows_linear")
    if sums:
        return RowSums(ws.view(torch.float32).view(-1, rows, n_out), (*x.shape[:-1], n_out), dtype)
    return out


class RowSums:
    """A product of a few rows still in its FP32 parts [splits, rows, n], for
    the norm that follows it (rms_norm_sums); ``tensor()`` is the product."""

    def __init__(self, parts: torch.Tensor, shape, dtype: torch.dtype) -> None:
        self.parts, self.shape, self.dtype = parts, torch.Size(shape), dtype

    def tensor(self) -> torch.Tensor:
        total = self.parts[0]
        for part in self.parts[1:]:  # in split order, as the kernels add
            total = total + part
        return total.to(self.dtype).view(self.shape)


def rms_norm_sums(x: RowSums, weight: torch.Tensor, eps: float, residual: torch.Tensor):
    """rms_norm(x.tensor(), weight, eps, residual) from the parts in one launch,
    or None for operands that the kernel does not take."""
    splits, rows, hidden = x.parts.shape
    size = x.dtype.itemsize
    if (weight.dtype != x.dtype or weight.shape != (hidden,) or residual.dtype != x.dtype
            or residual.shape != x.shape or hidden * size % 16 or hidden * size > 4096):
        return None
    rr, weight = _rows(residual, "residual"), weight.contiguous()
    if (rr.data_ptr() | weight.data_ptr()) & 15 or rr.stride(0) * size % 16 or rr.stride(0) < hidden:
        return None
    device = residual.device
    out, res_out = torch.empty((2, *x.shape), dtype=x.dtype, device=device)
    if (res_out.data_ptr() | x.parts.data_ptr()) & 15:
        return None
    with _lib.on(device):
        status = _lib.load().mlr_rms_norm_sums(
            x.parts.data_ptr(), splits, rr.data_ptr(), rr.stride(0), res_out.data_ptr(),
            weight.data_ptr(), out.data_ptr(), rows, hidden, float(eps),
            _lib.DTYPE_CODES[x.dtype], _lib.stream_handle(device))
    _lib.check(status, "mlr_rms_norm_sums")
    return out, res_out


def norm_silu_mul(x: torch.Tensor, residual: torch.Tensor, norm_weight: torch.Tensor, eps: float,
                  gate_up_weight: torch.Tensor):
    """(linear_silu_mul(n, gate_up_weight), r) for (n, r) = rms_norm(x,
    norm_weight, eps, residual) in one launch, or None for a call that
    mlr_norm_rows_linear does not take (16-bit types, at most 32 rows of at most
    1024)."""
    dtype, k = x.dtype, x.shape[-1]
    if (dtype not in (torch.bfloat16, torch.float16) or not x.is_cuda or _transformed()
            or k % 8 or k == 0
            or gate_up_weight.ndim != 2 or gate_up_weight.shape[1] != k
            or gate_up_weight.shape[0] % 2):
        return None
    rows, n = x.numel() // k, gate_up_weight.shape[0] // 2
    if (rows == 0 or rows > 32 or k > (1024 if rows <= 16 else 1008)
            or 2 * n * k * 2 > _ROWS_LIMIT[True, rows > 16, True]
            or x.shape != residual.shape or norm_weight.shape != (k,)):
        return None
    for t in (x, residual, norm_weight, gate_up_weight):
        if (t.dtype != dtype or t.device != x.device or t.stride(-1) != 1
                or type(t) not in (torch.Tensor, nn.Parameter) or t.data_ptr() & 15):
            return None
    if not gate_up_weight.is_contiguous():
        return None
    if torch.is_grad_enabled() and (x.requires_grad or residual.requires_grad
                                    or norm_weight.requires_grad):
        return None
    xr, rr = x.reshape(rows, k), residual.reshape(rows, k)
    xs, rs = (xr.stride(0), rr.stride(0)) if rows > 1 else (k, k)
    if xs < k or rs < k or xs % 8 or rs % 8 or (xr.data_ptr() | rr.data_ptr()) & 15:
        return None
    device = x.device
    out = torch.empty((*x.shape[:-1], n), dtype=dtype, device=device)
    res_out = torch.empty(x.shape, dtype=dtype, device=device)
    with _lib.on(device):
        status = _lib.load().mlr_norm_rows_linear(
            xr.data_ptr(), xs, rr.data_ptr(), rs, res_out.data_ptr(), norm_weight.data_ptr(),
            float(eps), gate_up_weight.data_ptr(), out.data_ptr(), n, rows, n, k,
            _lib.DTYPE_CODES[dtype], _lib.stream_handle(device))
    _lib.check(status, "mlr_norm_rows_linear")
    return out, res_out


def linear_silu_mul(x: torch.Tensor, gate_up_weight: torch.Tensor) -> torch.Tensor:
    """silu(x @ gate.T) * (x @ up.T) for the stacked weight [gate; up]
    [2 * intermediate, hidden]: one launch for a few rows, else the GEMM and
    silu_mul."""
    out = None
    if gate_up_weight.shape[0] % 2 == 0:
        out = _rows_linear(x, gate_up_weight, None, True)
    return silu_mul(F.linear(x, gate_up_weight)) if out is None else out


def plain(module: nn.Module, kind: type) -> bool:
    """Whether `module` is a `kind` that computes what its class says: no
    subclass, hook or replaced forward."""
    return (type(module) is kind and not module._forward_hooks
            and not module._forward_pre_hooks and not module._backward_hooks
            and not module._backward_pre_hooks and "forward" not in module.__dict__
            and not nn.modules.module._has_any_global_hook())


def apply_linear(module: nn.Module, x: torch.Tensor) -> torch.Tensor:
    """module(x) for a projection of the model: a plain nn.Linear over a few
    rows goes through mlr_rows_linear, anything else is called as it is."""
    if plain(module, nn.Linear):
        out = _rows_linear(x, module.weight, module.bias, False)
        if out is not None:
            return out
    return module(x)
