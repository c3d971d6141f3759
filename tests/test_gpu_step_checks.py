"""The one-launch metadata checks (mlr_check_step) against the torch
operations they replace, which still run for CPU tensors: the same error, or
none, for the same well- and ill-formed metadata."""

from __future__ import annotations

import random
from types import SimpleNamespace

import pytest
import torch

from mini_llm_runtime_amd import _lib
from mini_llm_runtime_amd.kernels import paged_attention as kpa
from mini_llm_runtime_amd.kernels import step_checks as kchk
from mini_llm_runtime_amd.model.qwen2 import TinyQwen2Model
from mini_llm_runtime_amd.model.qwen2_attention import Qwen2Attention
from mini_llm_runtime_amd.runtime import model_runner
from mini_llm_runtime_amd.runtime.paged_kv_cache import PagedKVCache
from mini_llm_runtime_amd.runtime.request import RequestStatus

pytestmark = pytest.mark.gpu
BS, BLOCKS = 16, 700


def _metadata(rng, reqs, decode_only, long_one=0, longest=90):
    """A well-formed step: {name: CPU tensor} and the requests' phases."""
    free = list(range(BLOCKS))
    rng.shuffle(free)
    tables, ctx, counts, phases = [], [], [], []
    for i in range(reqs):
        decode = decode_only or rng.random() < 0.5
        n = long_one if i == 0 and long_one else rng.randint(1, longest)
        count = 1 if decode and not (i == 0 and long_one) else rng.randint(1, n)
        if i == 0 and long_one:
            count, decode = n, False
        ctx.append(n)
        counts.append(count)
        phases.append(RequestStatus.DECODING if decode else RequestStatus.PREFILLING)
        tables.append([free.pop() for _ in range(-(-n // BS))])
    width = max(len(t) for t in tables) + rng.randint(0, 2)
    pos = [p for c, n in zip(counts, ctx) for p in range(n - c, n)]
    own = [i for i, c in enumerate(counts) for _ in range(c)]
    slots = [tables[i][p // BS] * BS + p % BS for i, p in zip(own, pos)]
    qsl = [0]
    for c in counts:
        qsl.append(qsl[-1] + c)
    t = {"tables": torch.tensor([x + [-1] * (width - len(x)) for x in tables]),
         "ctx": torch.tensor(ctx), "qsl": torch.tensor(qsl), "pos": torch.tensor(pos),
         "slots": torch.tensor(slots)}
    return t, phases


def _corrupt(rng, t, first=0):
    """Change one entry, of request `first` or a later one."""
    start = {"tables": first * t["tables"].shape[1], "ctx": first, "qsl": first}
    name = rng.choice(["tables", "ctx", "qsl", "pos", "slots", "repeat", "none"])
    if name == "none":
        return
    if name == "repeat":
        if len(t["slots"]) > 1:
            i, j = rng.sample(range(len(t["slots"])), 2)
            i = max(i, _first_token(t, first))
            t["slots"][i] = t["slots"][j]
        return
    flat = t[name].view(-1)
    i = rng.randrange(start.get(name, _first_token(t, first)), len(flat))
    flat[i] = rng.choice([-1, 0, -7, int(flat[i]) + 1, int(flat[i]) - 1, 2 ** 40, BLOCKS,
                          BLOCKS * BS, int(flat[rng.randrange(len(flat))])])


def _first_token(t, request):
    return min(max(int(t["qsl"][request]), 0), len(t["slots"]) - 1)


def _outcome(f):
    try:
        return repr(f())
    except (ValueError, IndexError) as e:
        return f"{type(e).__name__}: {e}"


def _same(device, t, f):
    want = _outcome(lambda: f({k: v.clone() for k, v in t.items()}))
    got = _outcome(lambda: f({k: v.to(device) for k, v in t.items()}))
    assert got == want
    return want


@pytest.mark.parametrize("reqs", [1, 2, 17, 300])
def test_same_errors_as_the_torch_checks(device, reqs):
    rng = random.Random(reqs)
    cache = SimpleNamespace(block_size=BS, num_blocks=BLOCKS)
    seen = set()
    # 300 requests of one or two blocks are more than the launch's workgroups
    # (256): rows from 256 on are second rows, and are corrupted on their own.
    many = reqs > 256
    for trial in range(60 if many else 150):
        decode_only = trial % 3 == 0
        t, phases = _metadata(rng, reqs, decode_only, longest=30 if many else 90)
        assert len(t["ctx"]) == reqs and kchk._lib.load().mlr_check_step_groups(
            reqs, len(t["slots"])) == max(min(reqs, 256), -(-len(t["slots"]) // 64))
        for _ in range(rng.randint(0, 2)):
            _corrupt(rng, t, first=257 if many and trial % 2 else 0)
        seen.add(_same(device, t, lambda m: kpa._validate_tables(m["tables"], m["ctx"], BS,
                                                                 BLOCKS)))
        if decode_only and len(t["pos"]) == len(t["ctx"]):
            seen.add(_same(device, t, lambda m: Qwen2Attention._check_decode_metadata(
                cache, m["pos"][:, None], m["slots"], m["tables"], m["ctx"])))
        for most in (90, 40):
            seen.add(_same(device, t, lambda m: TinyQwen2Model._check_packed_metadata(
                cache, m["pos"], m["slots"], m["tables"], m["qsl"], m["ctx"], most,
                len(m["pos"]))))

        def step(m):
            dev = m["pos"].device
            batch = model_runner.ModelBatch(
                [f"r{i}" for i in range(len(phases))], torch.zeros_like(m["pos"]), m["pos"],
                m["qsl"], phases, m["ctx"], m["tables"], m["slots"])
            weight = torch.zeros(1, device=dev)
            model = SimpleNamespace(parameters=lambda: iter([weight]))
            pool = SimpleNamespace(block_size=BS, num_blocks=BLOCKS, device=dev,
                                   dtype=weight.dtype)
            return model_runner._check_batch(model, batch, pool)

        seen.add(_same(device, t, step))
    assert len(seen) > 3


@pytest.mark.parametrize("tokens", [1, 63, 64, 65, 257, 1025, 1089, 8192, 8193])
def test_repeated_and_out_of_range_slots(device, tokens):
    rng = random.Random(tokens)
    caches = [PagedKVCache(1, 600, 16, 1, 8, device=d) for d in ("cpu", device)]
    good = rng.sample(range(9600), tokens)
    for edit in ({}, {tokens - 1: good[0]}, {0: -1}, {tokens // 2: 9600}, {tokens - 1: 9599}):
        slots = list(good)
        for i, v in edit.items():
            slots[i] = v
        for dtype in (torch.int64, torch.int32):
            got = [_outcome(lambda: c.check_slots(torch.tensor(slots, dtype=dtype).to(c.device)))
                   for c in caches]
            assert got[0] == got[1]
    assert (kchk.step_flags(16, 600, slots=torch.tensor(good).to(device)) is None) == (tokens > 8192)


def test_long_packed_step_and_strided_tables(device):
    """Requests over several workgroups' tokens, tables as a slice of wider ones."""
    t, _ = _metadata(random.Random(5), 60, False, long_one=5000)
    wide = torch.full((60, t["tables"].shape[1] + 5), -9)
    wide[:, :-5] = t["tables"]
    t["tables"] = wide
    cache = SimpleNamespace(block_size=BS, num_blocks=BLOCKS)

    def check(m):
        return TinyQwen2Model._check_packed_metadata(
            cache, m["pos"], m["slots"], m["tables"][:, :-5], m["qsl"], m["ctx"], 5000,
            len(m["pos"]))

    assert _same(device, t, check) == "None"
    t["slots"][-1] = t["slots"][700]
    assert "slot_mapping must match" in _same(device, t, check)


def test_entry_point_refuses_bad_arguments(device):
    lib = _lib.load()
    out = torch.zeros(8, dtype=torch.long, device=device)
    ctx = torch.ones(2, dtype=torch.long, device=device)

    def call(stride=2, width=2, reqs=2, tokens=0, bs=16, length=8, qsl=None, detail=0):
        return lib.mlr_check_step(out.data_ptr(), stride, width, ctx.data_ptr(), reqs, qsl, None,
                                  None, tokens, None, bs, 8, 0, detail, out.data_ptr(), length,
                                  _lib.stream_handle(device))

    assert call(stride=1) and call(bs=0) and call(length=1) and call(tokens=2) and call(detail=1)
    assert call(tokens=9000) and lib.mlr_check_step_groups(1, 8193) == 0
