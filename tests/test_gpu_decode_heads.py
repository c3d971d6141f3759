"""Decode at head sizes other than 64 and 128: the padded matrix-core kernel
against the generic kernel (which a split of 24 tokens still takes) and
against attention in 64 bits.

Both kernels round each score to the input type, as the reference does; their
FP32 sums run in another order, so a score may round to its neighbour: one
unit (2^-8 bf16, 2^-11 fp16 relative) of a score of up to about 6 moves its
probability by that much. Outputs are weighted means of |V| < 5, so 2e-2 holds
them for 16-bit types, and 1e-5 for FP32, the bounds of the other head sizes.
Against 64 bits the two kernels' errors are sums of independent roundings in
different orders: over 60 draws of one query their ratio is 0.54 to 1.001 in the
mean and scatters by up to 0.3 in FP32 at 20 keys, 0.01 in 16 bits. Over a case's
rows together the padded kernel may be 10% further off in one draw."""

from __future__ import annotations

import math

import pytest
import torch

from mini_llm_runtime_amd import _lib
from mini_llm_runtime_amd.kernels import paged_attention as kpa

pytestmark = pytest.mark.gpu
DTYPES = [torch.bfloat16, torch.float16, torch.float32]


def _case(dtype, d, hq, hkv, bs, lens, seed):
    gen = torch.Generator().manual_seed(seed)
    need = [-(-n // bs) for n in lens]
    perm = torch.randperm(sum(need) + 3, generator=gen).tolist()
    kc = torch.full((sum(need) + 3, bs, hkv, d), float("nan"), dtype=dtype)
    vc = kc.clone()
    tables, at = [], 0
    for n, nb in zip(lens, need):
        tables.append(perm[at:at + nb])
        at += nb
        pos = torch.arange(n)
        blocks = torch.tensor(tables[-1])[pos // bs]
        kc[blocks, pos % bs] = torch.randn(n, hkv, d, generator=gen).to(dtype)
        vc[blocks, pos % bs] = torch.randn(n, hkv, d, generator=gen).to(dtype)
    q = torch.randn(len(lens), hq, d, generator=gen).to(dtype)
    bt = torch.tensor([t + [-1] * (max(need) - len(t)) for t in tables])
    return q, kc, vc, bt, tables


def _exact(q, kc, vc, tables, lens):
    out = []
    for i, (t, n) in enumerate(zip(tables, lens)):
        k, v = (c[torch.tensor(t)].flatten(0, 1)[:n].double() for c in (kc, vc))
        group = q.shape[1] // k.shape[1]
        k, v = (x.repeat_interleave(group, dim=1) for x in (k, v))
        s = (q[i].double()[None] * k).sum(-1) / math.sqrt(q.shape[2])
        out.append((torch.softmax(s, dim=0)[..., None] * v).sum(0))
    return torch.stack(out)


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda t: str(t)[6:])
@pytest.mark.parametrize("d,hq,hkv,bs,lens", [
    (8, 4, 2, 16, [1, 40, 333]), (16, 4, 2, 16, [5] * 40), (24, 6, 6, 32, [64, 65, 1000]),
    (32, 6, 3, 16, [300] * 50), (56, 16, 1, 64, [2000, 17]), (72, 4, 4, 16, [700, 1, 129]),
    (80, 10, 2, 16, [2011, 103, 900]), (96, 8, 2, 16, [4000] * 3 + [7]), (120, 3, 1, 16, [513])])
def test_padded_heads_match_generic_and_float64(device, dtype, d, hq, hkv, bs, lens):
    q, kc, vc, bt, tables = _case(dtype, d, hq, hkv, bs, lens, seed=d)
    wide = torch.zeros(len(lens), hq, d + 8, dtype=dtype)
    wide[..., :d] = q
    args = (kc.to(device), vc.to(device), bt.to(device), torch.tensor(lens).to(device))
    got = kpa.paged_decode_launch(wide.to(device)[..., :d], *args)
    again = kpa.paged_decode_launch(q.to(device), *args)
    assert torch.equal(got, again)  # and the workspace came back zero
    generic = kpa.paged_decode_launch(q.to(device), *args, tokens_per_split=24)
    assert not any(w.any() for w in kpa._WORKSPACES.values())
    tol = 1e-5 if dtype is torch.float32 else 2e-2
    assert (got.double() - generic.double()).abs().max().item() <= tol
    want = _exact(q, kc, vc, tables, lens)
    off, was = ((x.double().cpu() - want).norm().item() for x in (got, generic))
    assert off <= 1.1 * was + 1e-6 * want.norm().item()
    for split in (16, 64, 512):
        other = kpa.paged_decode_launch(q.to(device), *args, tokens_per_split=split)
        assert (other.double() - got.double()).abs().max().item() <= tol


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda t: str(t)[6:])
@pytest.mark.parametrize("d,hq,hkv", [(16, 4, 2), (40, 5, 1), (96, 8, 2), (120, 4, 4)])
def test_append_equals_write_then_decode(device, dtype, d, hq, hkv):
    lens = [1, 16, 17, 700]
    q, kc, vc, bt, tables = _case(dtype, d, hq, hkv, 16, lens, seed=d + 1)
    gen = torch.Generator().manual_seed(9)
    new_k, new_v = (torch.randn(4, hkv, d, generator=gen).to(dtype).to(device) for _ in range(2))
    slots = torch.tensor([t[(n - 1) // 16] * 16 + (n - 1) % 16 for t, n in zip(tables, lens)])
    ctx, bt, q = torch.tensor(lens).to(device), bt.to(device), q.to(device)
    pools = [(kc.to(device), vc.to(device)) for _ in range(2)]
    got = kpa.paged_decode_launch(q, *pools[0], bt, ctx, new_k=new_k, new_v=new_v,
                                  slot_mapping=slots.to(device))
    for pool, rows in zip(pools[1], (new_k, new_v)):
        pool.view(-1, hkv, d)[slots.to(device)] = rows
    want = kpa.paged_decode_launch(q, *pools[1], bt, ctx)
    assert torch.equal(got, want)
    for a, b in zip(*pools):
        assert torch.equal(a.nan_to_num(9.0), b.nan_to_num(9.0))


def test_out_of_range_block_and_refusals(device):
    q, kc, vc, bt, _ = _case(torch.float16, 80, 4, 2, 16, [100, 100], seed=1)
    bt[0, 3] = kc.shape[0] + 5
    args = (q.to(device), kc.to(device), vc.to(device), bt.to(device),
            torch.tensor([100, 100]).to(device))
    got = kpa.paged_decode_launch(*args)
    generic = kpa.paged_decode_launch(*args, tokens_per_split=24)
    assert (got.double() - generic.double()).abs().max().item() <= 2e-2
    for split in (528, 1024):  # the generic kernel's limit stays these sizes' limit
        with pytest.raises(_lib.KernelError):
            kpa.paged_decode_launch(*args, tokens_per_split=split)


def test_scratch_limit_stays_the_generic_kernels(device, monkeypatch):
    """8,192-token tables: the generic default asks for 32 splits, the padded
    kernel uses 16; a workspace that was too small stays refused."""
    q, kc, vc, bt, _ = _case(torch.float16, 80, 4, 2, 16, [100, 33], seed=2)
    bt = torch.nn.functional.pad(bt, (0, 512 - bt.shape[1]), value=-1)
    args = (q.to(device), kc.to(device), vc.to(device), bt.to(device),
            torch.tensor([100, 33]).to(device))
    need = kpa.decode_workspace_bytes(2, 4, 80, 8192, torch.float16, 0)
    want = kpa.paged_decode_launch(*args)
    ws = torch.zeros(need, dtype=torch.uint8, device=device)
    assert torch.equal(kpa.paged_decode_launch(*args, workspace=ws), want)
    monkeypatch.setattr(_lib.load(), "mlr_paged_decode_workspace_size", lambda *a: 0)
    with pytest.raises(_lib.KernelError, match="smaller than"):  # the C entry's own check
        kpa.paged_decode_launch(*args, workspace=ws[:need - 256])


def _close_with_nonfinite(got, want, tol):
    got, want = got.double().cpu(), want.double().cpu()
    for same in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(same(got), same(want))
    fine = torch.isfinite(want)
    assert bool(fine.any()) and (got - want)[fine].abs().max().item() <= tol


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda t: str(t)[6:])
@pytest.mark.parametrize("d,hq,hkv", [(24, 4, 2), (80, 10, 2), (120, 3, 3)])
def test_infinite_values_as_in_float64(device, dtype, d, hq, hkv):
    """An infinite V gives that infinity, infinities of both signs NaN, at one
    token (p = 1) and among many."""
    lens = [1, 17, 40, 333, 700]
    q, kc, vc, bt, tables = _case(dtype, d, hq, hkv, 16, lens, seed=d)

    def put(b, token, dim, value):
        vc[tables[b][token // 16], token % 16, :, dim] = value

    put(0, 0, 0, math.inf)
    put(1, 16, 3, -math.inf)
    put(2, 5, 2, math.inf)
    put(2, 20, 2, -math.inf)  # both signs: NaN
    put(2, 7, 1, math.inf)
    put(2, 33, 1, math.inf)
    for token in range(0, 333, 9):
        put(3, token, d - 1, math.inf)
    put(4, 350, 5, math.nan)
    args = (q.to(device), kc.to(device), vc.to(device), bt.to(device),
            torch.tensor(lens).to(device))
    tol = 1e-5 if dtype is torch.float32 else 2e-2
    _close_with_nonfinite(kpa.paged_decode_launch(*args), _exact(q, kc, vc, tables, lens), tol)
    _close_with_nonfinite(kpa.paged_decode_launch(*args, tokens_per_split=24),
                          _exact(q, kc, vc, tables, lens), tol)


def _one_query(dtype, d, scores, values):
    """One request and head per row of scores [B, T]: q = (1, 0, ..), K rows whose
    first element gives those scores after the scale, V = values [B, T] in dim 1;
    (operands, the scores as rounded to dtype twice, in 64 bits)."""
    batch, tokens = scores.shape
    blocks = -(-tokens // 16)
    kc = torch.zeros(batch * blocks, 16, 1, d, dtype=dtype)
    vc = torch.zeros_like(kc)
    k0 = (scores * math.sqrt(d)).to(dtype)
    pad = blocks * 16 - tokens
    kc[..., 0, 0] = torch.nn.functional.pad(k0, (0, pad)).view(-1, 16)
    vc[..., 0, 1] = torch.nn.functional.pad(values.to(dtype), (0, pad)).view(-1, 16)
    q = torch.zeros(batch, 1, d, dtype=dtype)
    q[..., 0] = 1
    scale = torch.tensor(1 / math.sqrt(d), dtype=torch.float32)
    rounded = (k0.float() * scale).to(dtype).double()
    return q, kc, vc, torch.arange(batch * blocks).view(batch, blocks), rounded


@pytest.mark.parametrize("d", [40, 96])
def test_small_probabilities_count(device, d):
    """fp16: 999 probabilities of 2^-26 with V = 60,000 beside a larger key with
    V = 0. Half the smallest fp16 is 2^-25: as 16-bit parts they vanish."""
    scores = torch.full((1, 1000), -18.0)
    scores[0, 500] = 0
    values = torch.full((1, 1000), 60000.0)
    values[0, 500] = 0
    q, kc, vc, bt, rounded = _one_query(torch.float16, d, scores, values)
    p = torch.softmax(rounded, dim=1)
    want = (p * values.double()).sum().item()
    got = kpa.paged_decode_launch(q.to(device), kc.to(device), vc.to(device), bt.to(device),
                                  torch.tensor([1000]).to(device))[0, 0, 1].item()
    # fp16 rounding 2^-11, and FP32 exponents of 18 * log2(e) = 26 +- 26 * 2^-24.
    assert 0.4 < want and abs(got - want) <= 1e-3 * want


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda t: str(t)[6:])
@pytest.mark.parametrize("d", [40, 96])
def test_probabilities_keep_24_bits(device, dtype, d):
    """Keys of score s, s and s beside one of score 0 with V chosen to cancel:
    1 - p v1 - p v2 is about 2^-16 of the sum, where an error of 2^-18 in p shows.
    FP32 leaves 2^-24 in p (exp2 to one unit, its argument s log2(e) of up to 2 to
    half of one) and in each sum: 6 of them, 4e-7; 2^-8 is the output."""
    batch = 64
    s = torch.linspace(-1.3, -0.05, batch)[:, None]
    scores = torch.cat([torch.zeros(batch, 1), s.expand(batch, 2)], dim=1)
    rounded = _one_query(dtype, d, scores, torch.zeros(batch, 3))[4]
    p = rounded.exp()[:, 1]
    v1 = (1 / p).to(dtype).double()
    rest = 1 - p * v1
    # The last key takes what is left but for about 2^-15.
    v2 = ((rest - 2.0 ** -15) / p).to(dtype).double()
    values = torch.stack([torch.ones(batch).double(), -v1, -v2], dim=1)
    q, kc, vc, bt, rounded = _one_query(dtype, d, scores, values)
    want = (rounded.exp() * values).sum(1) / rounded.exp().sum(1)
    got = kpa.paged_decode_launch(q.to(device), kc.to(device), vc.to(device), bt.to(device),
                                  torch.full((batch,), 3).to(device))[:, 0, 1].double().cpu()
    assert want.abs().min().item() > 2.0 ** -18
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 4e-7).all()


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda t: str(t)[6:])
@pytest.mark.parametrize("d,hq,hkv", [(24, 4, 2), (80, 10, 2)])
def test_scores_of_minus_infinity(device, dtype, d, hq, hkv):
    """Keys whose scores pass the type's range, alone in a 16-token tile or all
    of a split: -inf takes no weight, +inf makes the output NaN, as on the
    generic kernel (and in 64 bits with the scores so rounded)."""
    lens = [1, 17, 18, 333, 700]
    q, kc, vc, bt, tables = _case(dtype, d, hq, hkv, 16, lens, seed=d + 7)

    def key(b, tokens, value):
        for t in tokens:
            kc[tables[b][t // 16], t % 16] = 0
            kc[tables[b][t // 16], t % 16, :, 1] = value

    q[:, :, 1] = q[:, :, 1].abs() + 2
    q[2, 0, 1] *= -1  # this head's scores are +inf
    big = 60000.0 if dtype is torch.float16 else 3e38
    key(0, [0], -big)
    key(1, [16], -big)
    key(2, [17], -big)
    key(3, range(0, 330), -big)
    key(4, range(0, 64), -big)
    key(4, [699], -big)
    args = (q.to(device), kc.to(device), vc.to(device), bt.to(device),
            torch.tensor(lens).to(device))
    got = kpa.paged_decode_launch(*args)
    tol = 1e-5 if dtype is torch.float32 else 2e-2
    _close_with_nonfinite(got, kpa.paged_decode_launch(*args, tokens_per_split=24), tol)
    assert got[0].isnan().all() and got[2, 0].isnan().all()
    assert torch.isfinite(got[[1, 3, 4]]).all() and torch.isfinite(got[2, 1:]).all()
    assert not any(w.any() for w in kpa._WORKSPACES.values())


def test_whole_splits_of_out_of_range_blocks(device):
    """Block ids out of range over whole splits, the first and the last ones."""
    lens = [700, 700, 1500]
    q, kc, vc, bt, _ = _case(torch.bfloat16, 80, 10, 2, 16, lens, seed=3)
    bt[0, :30] = -5
    bt[1, 20:44] = kc.shape[0] + 1
    bt[2, :80] = 2 ** 40
    args = (q.to(device), kc.to(device), vc.to(device), bt.to(device),
            torch.tensor(lens).to(device))
    for split in (0, 64, 256):
        got = kpa.paged_decode_launch(*args, tokens_per_split=split)
        _close_with_nonfinite(got, kpa.paged_decode_launch(*args, tokens_per_split=24), 2e-2)
        assert torch.isfinite(got).all()
