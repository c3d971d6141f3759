"""Prefill calls whose key ranges are split over workgroups against the same
calls unsplit.

Both forms compute the same FP32 scores and sums; they differ in the reference
point of each probability's exponent, so each probability is rounded to the
16-bit operand at another scale (u relative, u = 2^-8 bf16, 2^-11 fp16, in
each form), in the order of FP32 sums, and in the final rounding (u each):
|split - unsplit| <= 2 u (max |V| + |y|), with 1% for the FP32 terms.
"""

from __future__ import annotations

import pytest
import torch

from mini_llm_runtime_amd import _lib
from mini_llm_runtime_amd.kernels import paged_attention as kpa

pytestmark = pytest.mark.gpu

ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _pool(lens, hkv, d, bs, dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    need = [-(-n // bs) for n in lens]
    perm = torch.randperm(sum(need) + 2, generator=gen).tolist()
    kc = torch.full((sum(need) + 2, bs, hkv, d), float("nan"), dtype=dtype)
    vc, tables, at = kc.clone(), [], 0
    for n, nb in zip(lens, need):
        tables.append(perm[at:at + nb])
        at += nb
        pos = torch.arange(n)
        blocks = torch.tensor(tables[-1])[pos // bs]
        kc[blocks, pos % bs] = torch.randn(n, hkv, d, generator=gen).to(dtype)
        vc[blocks, pos % bs] = torch.randn(n, hkv, d, generator=gen).to(dtype)
    return kc, vc, tables, gen


def _both(monkeypatch, call, splits: bool):
    seen = []
    workspace = kpa._prefill_workspace
    monkeypatch.setattr(kpa, "_prefill_workspace",
                        lambda *a: seen.append(workspace(*a)) or seen[-1])
    got = call().double().cpu()
    monkeypatch.setattr(kpa, "_prefill_workspace", lambda *a: (None, 0))
    want = call().double().cpu()
    monkeypatch.undo()
    assert (seen[0][1] > 0) == splits
    return got, want


def _close(got, want, vc, dtype):
    vmax = float(torch.nan_to_num(vc.float()).abs().max())
    assert bool(torch.isfinite(got).all())
    assert bool(((got - want).abs() <= 2.02 * ULP[dtype] * (vmax + want.abs())).all())


@pytest.mark.parametrize("dtype", list(ULP), ids=lambda t: str(t)[6:])
@pytest.mark.parametrize("hq,hkv,d,prefix,chunk,splits", [
    (14, 2, 64, 1664, 64, False),     # 27 tiles: too few to pay for the merge
    (14, 2, 64, 1665, 64, True),      # 28 tiles
    (14, 2, 64, 5000, 129, True), (28, 4, 128, 4000, 500, True), (4, 1, 128, 2100, 1, True),
    (8, 2, 96, 3000, 200, True),
    (32, 8, 128, 3000, 1024, False)])  # a workgroup per CU without a split
def test_chunk_split_equals_unsplit(device, monkeypatch, dtype, hq, hkv, d, prefix, chunk, splits):
    context = prefix + chunk
    kc, vc, tables, gen = _pool([context], hkv, d, 16, dtype, prefix)
    q = torch.randn(chunk, hq, d, generator=gen).to(dtype).to(device)
    k, v = kc.to(device), vc.to(device)
    got, want = _both(monkeypatch, lambda: kpa.paged_attention_prefill_chunk_tiled(
        q, k, v, tables[0], prefix, context, 16, 64), splits)
    _close(got, want, vc, dtype)


@pytest.mark.parametrize("dtype", list(ULP), ids=lambda t: str(t)[6:])
@pytest.mark.parametrize("hq,hkv,d,prefix,chunk,splits", [
    (8, 2, 96, 256, 64, False),  # 5 tiles
    (8, 2, 96, 257, 64, True),   # 6 tiles, in parts of 3
    (6, 3, 32, 448, 64, True),   # 8 tiles in parts of 4
    (4, 2, 16, 1000, 9, True), (5, 1, 80, 640, 129, True),
    (32, 8, 96, 900, 640, False)])  # a workgroup per CU without a split
def test_padded_heads_split_equals_unsplit(device, monkeypatch, dtype, hq, hkv, d, prefix, chunk,
                                           splits):
    test_chunk_split_equals_unsplit(device, monkeypatch, dtype, hq, hkv, d, prefix, chunk, splits)


@pytest.mark.parametrize("dtype", list(ULP), ids=lambda t: str(t)[6:])
def test_ragged_varlen_split_equals_unsplit(device, monkeypatch, dtype):
    """Items with one split, several, and none (query tiles past a chunk), and
    an out-of-range block inside one split."""
    seqs = [(0, 5), (3000, 140), (700, 33), (0, 300)]
    hq, hkv, d, bs = 4, 2, 64, 32
    lens = [p + n for p, n in seqs]
    kc, vc, tables, gen = _pool(lens, hkv, d, bs, dtype, 3)
    tables[1][50] = kc.shape[0] + 7
    width = max(len(t) for t in tables)
    bt = torch.tensor([t + [-1] * (width - len(t)) for t in tables]).to(device)
    rows = [n for _, n in seqs]
    qsl = torch.tensor([sum(rows[:i]) for i in range(len(rows) + 1)]).to(device)
    q = torch.randn(sum(rows), hq, d, generator=gen).to(dtype).to(device)
    k, v = kc.to(device), vc.to(device)
    got, want = _both(monkeypatch, lambda: kpa.paged_attention_prefill_varlen(
        q, k, v, bt, qsl, torch.tensor(lens).to(device), bs), True)
    _close(got, want, vc, dtype)


def test_small_workspace_runs_unsplit(device):
    lib = _lib.load()
    assert lib.mlr_paged_prefill_workspace_size(1, 64, 4096, 14, 64, 2) > 0
    for args in ((1, 64, 512, 14, 64, 2), (64, 512, 4096, 14, 64, 2), (1, 64, 4096, 14, 64, 0),
                 (1, 64, 4096, 14, 60, 2), (0, 64, 4096, 14, 64, 2)):
        assert lib.mlr_paged_prefill_workspace_size(*args) == 0
