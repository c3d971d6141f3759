"""What the Python entry points hand to the HIP library, on the CPU: a stand-in
library records the calls, so a form that the kernels must refuse or never see
is shown without a GPU."""

from __future__ import annotations

import contextlib

import numpy as np
import pytest
import torch

from mini_llm_runtime_amd import _lib
from mini_llm_runtime_amd.kernels import layer_ops as kops
from mini_llm_runtime_amd.kernels import paged_attention as kpa


@pytest.fixture
def calls(monkeypatch):
    """[(entry point, arguments)] of the library calls a test makes."""
    seen = []

    class Library:
        def __getattr__(self, name):
            def entry(*args):
                seen.append((name, args))
                return 0

            return entry

    monkeypatch.setattr(_lib, "load", Library)
    monkeypatch.setattr(_lib, "on", lambda device: contextlib.nullcontext())
    monkeypatch.setattr(_lib, "stream_handle", lambda device: 0)
    monkeypatch.setattr(_lib, "require_hip", lambda *tensors, what: tensors[0].device)
    monkeypatch.setattr(kops, "supported", lambda x: x.dtype in kops.DTYPES)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    return seen


@pytest.mark.parametrize("strided", ["x", "residual", "neither"])
def test_rms_norm_passes_a_zero_row_stride_on(calls, strided):
    """One row expanded over many has row stride 0, which the entry point
    refuses; read as whole rows it would run past the buffer."""
    row = torch.ones(1, 64)
    x, residual = (row.expand(4, 64) if strided == name else torch.ones(4, 64)
                   for name in ("x", "residual"))
    kops.rms_norm(x, torch.ones(64), 1e-6, residual=residual)
    (name, args), = calls
    assert name == "mlr_rms_norm"
    assert (args[1], args[3]) == (0 if strided == "x" else 64, 0 if strided == "residual" else 64)


@pytest.mark.gpu
@pytest.mark.parametrize("strided", ["x", "residual"])
def test_rms_norm_refuses_a_zero_row_stride(device, strided):
    row = torch.ones(1, 64, device=device)
    x, residual = (row.expand(4, 64) if strided == name else torch.ones(4, 64, device=device)
                   for name in ("x", "residual"))
    with pytest.raises(_lib.KernelError, match="row stride"):
        kops.rms_norm(x, torch.ones(64, device=device), 1e-6, residual=residual)


@pytest.mark.parametrize("eps", [1e-6, np.float32(1e-6), torch.tensor(1e-6), 1])
def test_norms_take_any_number_as_eps(calls, eps):
    """The library takes a C double, which ctypes makes of int and float only."""
    kops.rms_norm(torch.ones(4, 64), torch.ones(64), eps)
    kops.rms_norm_sums(kops.RowSums(torch.zeros(2, 4, 64), (4, 64), torch.float32),
                       torch.ones(64), eps, torch.ones(4, 64))
    assert [name for name, _ in calls] == ["mlr_rms_norm", "mlr_rms_norm_sums"]
    for _, args in calls:
        assert float(eps) in [a for a in args if type(a) is float]


@pytest.mark.parametrize("entries,want", [
    ([3, 1, 2 ** 70], [3, 1]),  # past the blocks in use: any number
    ([3, 1, -2 ** 70], [3, 1]), ([3, 1, 99], [3, 1]), ([3, 1.0, -1.5], [3, 1]),
    ([3, 2 ** 70, 1], None), ([1e300, 3, 1], None), ([3, -1, 1], None), ([3, 8, 1], None),
    ([torch.tensor(3), torch.tensor(1), torch.tensor(-4)], [3, 1]),
    ([torch.tensor(3.0), torch.tensor(1.0), torch.tensor(-4.0)], [3, 1])])
def test_host_tables_beyond_the_blocks_in_use(calls, entries, want):
    """Only the blocks that the context uses are looked at for range."""
    def chunk():
        kv = torch.zeros(8, 16, 1, 8)
        return kpa.paged_attention_prefill_chunk_tiled(torch.zeros(4, 1, 8), kv, kv, entries, 20,
                                                       24, 16, 64)

    if want is None:
        with pytest.raises(ValueError, match="out-of-range physical block"):
            chunk()
        return
    chunk()
    assert list(kpa._host_blocks(entries, 2, 8)) == want
    assert [a for a in calls if a[0] == "mlr_stage_i64"][0][1][1] == 2


@pytest.mark.parametrize("max_query_len", [None, 4])
def test_varlen_refuses_a_scalar_query_start_loc(calls, max_query_len):
    """A 0-d query_start_loc holds one number where the kernel reads two."""
    kv = torch.zeros(8, 16, 1, 8)
    with pytest.raises(IndexError):
        kpa.paged_attention_prefill_varlen(
            torch.zeros(4, 1, 8), kv, kv, torch.zeros(1, 1, dtype=torch.long), torch.tensor(0),
            torch.tensor([4]), 16, max_query_len=max_query_len)
    assert not calls
