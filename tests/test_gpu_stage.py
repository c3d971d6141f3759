"""Host block tables staged as kernel arguments (mlr_stage_i64): exact values
at the launches' edges, in stream order, and what stays refused."""

from __future__ import annotations

from array import array

import numpy as np
import pytest
import torch

from mini_llm_runtime_amd import _lib
from mini_llm_runtime_amd.kernels import paged_attention as kpa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 959, 960, 961, 1920, 3839, 3840, 3841])
def test_values_arrive(device, n):
    values = [(i * 7919) % 2147483647 for i in range(n)]
    values[-1] = 2147483647
    assert kpa._device_ints(array("q", values), device).tolist() == values
    assert kpa._device_ints(array("q", [2 ** 31] * n), device).tolist() == [2 ** 31] * n


def test_lists_may_be_reused_at_once(device):
    """The list's memory is free when the call returns; a long kernel ahead of
    it on the stream does not change what arrives."""
    busy = torch.randn(4096, 4096, device=device)
    buf, got = array("q", [0] * 100), []
    for step in range(5):
        busy = busy @ busy * 1e-3
        for i in range(100):
            buf[i] = step * 100 + i
        got.append(kpa._device_ints(buf, device))
    for step, t in enumerate(got):
        assert t.tolist() == list(range(step * 100, step * 100 + 100))


def test_tables_of_any_integers(device):
    k = torch.randn(8, 16, 2, 64, device=device).half()
    v = torch.randn(8, 16, 2, 64, device=device).half()
    q = torch.randn(4, 64, device=device).half()
    want = kpa.paged_attention_decode(q, k, v, [3, 1, 5], 40, 16)
    for table in ([np.int64(3), np.int32(1), 5], np.array([3, 1, 5, -1]), [3, 1, 5, -1, 99],
                  [torch.tensor(3), 1, 5], (3, 1, 5)):
        assert torch.equal(kpa.paged_attention_decode(q, k, v, table, 40, 16), want)
    for bad in ([3, 8, 5], [3, -1, 5], [3, 2 ** 70, 5]):
        with pytest.raises(ValueError, match="out-of-range"):
            kpa.paged_attention_decode(q, k, v, bad, 40, 16)
    with pytest.raises(TypeError):
        kpa.paged_attention_decode(q, k, v, [3, None, 5], 40, 16)


def test_refused(device):
    lib = _lib.load()
    out = torch.zeros(8, dtype=torch.long, device=device)
    buf = array("q", [1, 2 ** 31])
    stream = _lib.stream_handle(device)
    assert lib.mlr_stage_i64(buf.buffer_info()[0], 2, out.data_ptr(), stream) != 0
    assert lib.mlr_stage_i64(buf.buffer_info()[0], 3841, out.data_ptr(), stream) != 0
    assert lib.mlr_stage_i64(None, 1, out.data_ptr(), stream) != 0
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=side):
        with pytest.raises(RuntimeError, match="captured"):
            kpa._device_ints(array("q", [1]), device)
        out.fill_(3)
    graph.replay()
    torch.cuda.synchronize()
    assert out.tolist() == [3] * 8
