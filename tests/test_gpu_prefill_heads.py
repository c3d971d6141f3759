"""Packed prefill at head sizes other than 64 and 128 against attention in 64
bits.

Bound per output: q.k of 16-bit inputs in FP32 is off by at most
(d + 2) * 2^-24 * sum |q||k| (under 2^-15 after the scale, for these inputs),
which moves a probability by that much relative; exp2 and the sums, FP32
probabilities times V, add a few 2^-22. The weighted mean of V is then off by
under 2^-14 max |V|, and the result is rounded once (2^-8 bf16, 2^-11 fp16).
FP32 inputs stay FP32 throughout: errors of independent roundings, about
sqrt(d) 2^-24 |q||k| in a score, stay under the 1e-5 that the FP32 paths are
held to.
"""

from __future__ import annotations

import math

import pytest
import torch

from mini_llm_runtime_amd.kernels import paged_attention as kpa

pytestmark = pytest.mark.gpu

HALF_ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}


def _slack(dtype, vmax):
    return 1e-5 if dtype is torch.float32 else 2.0 ** -14 * vmax


def _attend(q, k, v, prefix):
    group = q.shape[1] // k.shape[1]
    k, v = (t.repeat_interleave(group, dim=1).transpose(0, 1) for t in (k, v))
    scores = torch.matmul(q.transpose(0, 1), k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[2])
    seen = (torch.arange(k.shape[1], device=q.device)[None, :]
            <= prefix + torch.arange(q.shape[0], device=q.device)[:, None])
    probs = torch.softmax(scores.masked_fill(~seen, float("-inf")), dim=-1)
    return torch.matmul(probs, v.contiguous()).transpose(0, 1)


SHAPES = [(8, 4, 2, 16), (16, 4, 2, 16), (24, 6, 6, 32), (32, 6, 3, 16), (40, 5, 1, 16),
          (56, 4, 2, 64), (72, 4, 4, 16), (80, 10, 2, 16), (96, 8, 2, 16), (120, 3, 1, 32)]
# The 16-bit kernels pre-scale q at 64 and 128, another bound than this one.
CASES = [(t, *s) for t in HALF_ULP for s in SHAPES]
CASES += [(torch.float32, 64, 14, 2, 16), (torch.float32, 128, 4, 1, 16)]


@pytest.mark.parametrize("dtype,d,hq,hkv,bs", CASES, ids=lambda v: str(v).split(".")[-1])
def test_other_head_sizes_match_float64(device, dtype, d, hq, hkv, bs):
    gen = torch.Generator().manual_seed(d)
    seqs = [(0, 1), (130, 33), (0, 129), (700, 200), (15, 64)]  # (prefix, queries)
    need = [-(-(p + n) // bs) for p, n in seqs]
    perm = torch.randperm(sum(need) + 3, generator=gen).tolist()
    # Rows past each context hold NaN: nothing may read them into a product.
    kc = torch.full((sum(need) + 3, bs, hkv, d), float("nan"), dtype=dtype)
    vc = kc.clone()
    tables, want, qs, at = [], [], [], 0
    for (p, n), nb in zip(seqs, need):
        table = perm[at:at + nb]
        at += nb
        tables.append(table + [-1] * (max(need) - nb))
        k, v = (torch.randn(p + n, hkv, d, generator=gen).to(dtype) for _ in range(2))
        pos = torch.arange(p + n)
        blocks = torch.tensor(table)[pos // bs]
        kc[blocks, pos % bs], vc[blocks, pos % bs] = k, v
        q = torch.randn(n, hq, d, generator=gen).to(dtype)
        qs.append(q)
        want.append(_attend(q.double(), k.double(), v.double(), p))
    want = torch.cat(want)
    lens = [n for _, n in seqs]
    # q as rows of a wider buffer, as a view of a fused projection would be.
    wide = torch.full((sum(lens), hq, d + 8), 7.0, dtype=dtype)
    wide[..., :d] = torch.cat(qs)
    args = (kc.to(device), vc.to(device), torch.tensor(tables).to(device),
            torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)]).to(device),
            torch.tensor([p + n for p, n in seqs]).to(device), bs)
    got = kpa.paged_attention_prefill_varlen(wide.to(device)[..., :d], *args).double().cpu()
    vmax = float(torch.nan_to_num(vc.float()).abs().max())
    bound = HALF_ULP[dtype] * 1.01 * want.abs() + _slack(dtype, vmax)
    assert bool(((got - want).abs() <= bound).all()), ((got - want).abs() - bound).max()
    assert torch.equal(
        kpa.paged_attention_prefill_varlen(torch.cat(qs).to(device), *args).double().cpu(), got)


@pytest.mark.parametrize("seqs,longest,prefix,hq,hkv,d", [
    (16, 200, 0, 28, 4, 128),   # one wave per workgroup
    (10, 330, 60, 28, 4, 128),  # two
    (16, 180, 30, 14, 2, 64), (4, 300, 900, 14, 2, 64),  # four, items ranked
    (2, 40, 700, 4, 2, 32)])    # eight
def test_fp32_workgroup_shapes_match_float64(device, seqs, longest, prefix, hq, hkv, d):
    """FP32: every wave count of the launcher, ragged chunks and prefixes."""
    gen = torch.Generator().manual_seed(seqs)
    n = torch.randint(1, longest + 1, (seqs,), generator=gen).tolist()
    n[-1] = longest
    p = torch.randint(0, prefix + 1, (seqs,), generator=gen).tolist()
    need = [-(-(a + b) // 16) for a, b in zip(n, p)]
    perm = torch.randperm(sum(need), generator=gen).tolist()
    kc, vc = (torch.randn(sum(need), 16, hkv, d, generator=gen).to(device) for _ in range(2))
    q = torch.randn(sum(n), hq, d, generator=gen).to(device)
    tables = [perm[sum(need[:i]):sum(need[:i + 1])] for i in range(seqs)]
    bt = torch.tensor([t + [-1] * (max(need) - len(t)) for t in tables]).to(device)
    qsl = [sum(n[:i]) for i in range(seqs + 1)]
    ctx = [a + b for a, b in zip(n, p)]
    got = kpa.paged_attention_prefill_varlen(q, kc, vc, bt, torch.tensor(qsl).to(device),
                                             torch.tensor(ctx).to(device), 16)
    for i, t in enumerate(tables):
        k, v = (c[torch.tensor(t, device=device)].reshape(-1, hkv, d)[:ctx[i]].double()
                for c in (kc, vc))
        want = _attend(q[qsl[i]:qsl[i + 1]].double(), k, v, p[i])
        off = (got[qsl[i]:qsl[i + 1]].double() - want).abs().max().item()
        assert off <= 1e-5, (i, off)


@pytest.mark.parametrize("dtype", list(HALF_ULP), ids=lambda t: str(t)[6:])
@pytest.mark.parametrize("d", [24, 80])
@pytest.mark.parametrize("scale", [1e-50, 1e-40, 1e-29])
def test_scales_near_zero(device, dtype, d, scale):
    """A scale that rounds to 0 or a subnormal FP32 number weighs all keys that a
    query sees alike: the running mean of V."""
    gen = torch.Generator().manual_seed(d)
    n = 50
    k, v = (torch.randn(4, 16, 2, d, generator=gen).to(dtype) for _ in range(2))
    q = torch.randn(n, 4, d, generator=gen).to(dtype)
    got = kpa.paged_prefill_launch(
        q.to(device), k.to(device), v.to(device), torch.arange(4)[None].to(device),
        torch.tensor([0, n]).to(device), torch.tensor([n]).to(device), n, scale=scale)
    rows = v.view(64, 2, d)[:n].double().repeat_interleave(2, dim=1)
    want = rows.cumsum(0) / torch.arange(1, n + 1)[:, None, None]
    bound = HALF_ULP[dtype] * 1.01 * want.abs() + _slack(dtype, 5)
    assert bool(((got.double().cpu() - want).abs() <= bound).all())


def _one_chunk(device, q, k, v, prefix):
    """One sequence in 16-row blocks, in order: (its chunk prefill, the
    operands moved)."""
    n = k.shape[0]
    pools = []
    for t in (k, v):
        pool = torch.full((-(-n // 16) * 16, *t.shape[1:]), float("nan"), dtype=t.dtype)
        pool[:n] = t
        pools.append(pool.view(-1, 16, *t.shape[1:]).to(device))
    return kpa.paged_attention_prefill_chunk_tiled(
        q.to(device), *pools, list(range(pools[0].shape[0])), prefix, n, 16, 64)


@pytest.mark.parametrize("d", [40, 96])
@pytest.mark.parametrize("prefix", [999, 3999])  # whole, and split over workgroups
def test_small_probabilities_count(device, d, prefix):
    """fp16: probabilities of 2^-26 with V = 60,000 beside one larger key with
    V = 0. Half the smallest fp16 is 2^-25: as 16-bit parts they vanish."""
    k, v = (torch.zeros(prefix + 1, 1, d, dtype=torch.float16) for _ in range(2))
    q = torch.zeros(1, 1, d, dtype=torch.float16)
    q[..., 0] = 1
    k[:, 0, 0] = -18 * math.sqrt(d)
    k[500, 0, 0] = 0
    v[:, 0, 1] = 60000
    v[500, 0, 1] = 0
    scores = k[:, 0, 0].double() / math.sqrt(d)
    want = (torch.softmax(scores, 0) * v[:, 0, 1].double()).sum().item()
    got = _one_chunk(device, q, k, v, prefix)[0, 0, 1].item()
    # fp16 rounding 2^-11; FP32 scores of 18 move a probability by 18 * 2^-23.
    assert 0.4 < want and abs(got - want) <= 1e-3 * want


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda t: str(t)[6:])
@pytest.mark.parametrize("d", [40, 96])
def test_probabilities_keep_24_bits(device, dtype, d):
    """Keys of score s, s and s beside one of score 0 with V chosen to cancel:
    1 - p v1 - p v2 is about 2^-16 of the sum, where an error of 2^-18 in p shows.
    FP32 leaves 2^-23 in p (its score and exp2) and 2^-24 in each sum: 4e-7 in
    all; 2^-8 is the output."""
    for s in torch.linspace(-1.3, -0.05, 24).tolist():
        k, v = (torch.zeros(3, 1, d, dtype=dtype) for _ in range(2))
        q = torch.zeros(1, 1, d, dtype=dtype)
        q[..., 0] = 1
        k[1:, 0, 0] = s * math.sqrt(d)
        p = (k[1, 0, 0].double() / math.sqrt(d)).exp()
        v[0, 0, 1] = 1
        v[1, 0, 1] = -1 / p
        v[2, 0, 1] = -(1 + p * v[1, 0, 1].double() - 2.0 ** -15) / p
        want = (1 + p * v[1:, 0, 1].double().sum()) / (1 + 2 * p)
        got = _one_chunk(device, q, k, v, 2)[0, 0, 1].double().cpu()
        assert 2.0 ** -18 < abs(want)
        assert abs(got - want) <= 2.0 ** -8 * abs(want) + 4e-7, (s, got, want)


def _nonfinite_case(dtype, hq, hkv, d, prefix, n, seed):
    """q, k, v with infinities and NaN in V rows a sequence owns: behind the
    prefix, on the diagonal, next to each other and of both signs."""
    gen = torch.Generator().manual_seed(seed)
    q = torch.randn(n, hq, d, generator=gen).to(dtype)
    k, v = (torch.randn(prefix + n, hkv, d, generator=gen).to(dtype) for _ in range(2))
    last = prefix + n - 1
    for t, dim, value in ((last, 0, math.inf), (last - n // 2, 1, -math.inf),
                          (last - n // 3, 2, math.nan), (last - n // 3, 3, math.inf),
                          (last - n // 3 + 1, 3, -math.inf), (prefix, d - 1, math.inf),
                          (prefix // 2, 4, math.inf), (last - n // 5, d - 1, math.inf),
                          (last - n // 7, d // 2, -math.inf)):
        t = min(t, last)
        v[t, t % hkv, dim] = value
    return q, k, v


def _attend_nonfinite(q, k, v, prefix):
    """_attend where only the keys a query sees meet it."""
    return torch.cat([_attend(q[i:i + 1], k[:prefix + i + 1], v[:prefix + i + 1], prefix + i)
                      for i in range(q.shape[0])])


NONFINITE = [(t, d, *rest) for t in HALF_ULP for d in (24, 80, 96, 120)
             for rest in ((0, 75), (300, 1), (70, 160), (2500, 40))]
NONFINITE += [(torch.float32, d, *rest) for d in (16, 32, 64, 128)
              for rest in ((0, 75), (70, 160), (2500, 40))]


@pytest.mark.parametrize("dtype,d,prefix,n", NONFINITE, ids=lambda v: str(v).split(".")[-1])
def test_infinite_values_as_in_float64(device, dtype, d, prefix, n):
    """A value that is not finite reaches the queries that see its key, as that
    infinity or NaN, and no other query."""
    hq, hkv = 4, 2
    q, k, v = _nonfinite_case(dtype, hq, hkv, d, prefix, n, d + n)
    got = _one_chunk(device, q, k, v, prefix).double().cpu()
    want = _attend_nonfinite(q.double(), k.double(), v.double(), prefix)
    for same in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(same(got), same(want))
    fine = torch.isfinite(want)
    bound = HALF_ULP[dtype] * 1.01 * want.abs() + _slack(dtype, 5)
    assert fine.any() and bool(((got - want).abs() <= bound)[fine].all())
