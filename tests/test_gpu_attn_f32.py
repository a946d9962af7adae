"""The fp32 matrix-core attention kernel: row-tile edges, long contexts, and values that are not finite."""

from __future__ import annotations

import math
import random

import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


def _pool(gpu, hkv, d, bs, ends, seed):
    gen = torch.Generator(device=gpu).manual_seed(seed)
    need = [-(-e // bs) for e in ends]
    order = list(range(sum(need) + 3))
    random.Random(seed).shuffle(order)
    k = torch.randn(len(order), hkv, bs, d, generator=gen, device=gpu)
    v = torch.randn(len(order), hkv, bs, d, generator=gen, device=gpu)
    tab = torch.full((len(ends), max(need)), -7, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        tab[i, :n] = torch.tensor(order[at:at + n], dtype=torch.int32)
        at += n
    return k, v, tab.to(gpu), gen


def _exact(q, k, v, tab, starts, lengths, bs):
    """float64 causal attention of packed rows [N, Hq, D]."""
    out, at = torch.empty_like(q, dtype=torch.float64), 0
    g = q.shape[1] // k.shape[1]
    for i, (a, n) in enumerate(zip(starts, lengths)):
        end = a + n
        rows = tab[i, :-(-end // bs)].long()
        kk = k[rows].double().transpose(1, 2).reshape(-1, k.shape[1], k.shape[3])[:end]
        vv = v[rows].double().transpose(1, 2).reshape(-1, v.shape[1], v.shape[3])[:end]
        for t in range(n):
            for h in range(q.shape[1]):
                m = a + t + 1
                s = kk[:m, h // g] @ q[at + t, h].double() / math.sqrt(q.shape[2])
                p = torch.softmax(s, 0)
                vis = vv[:m, h // g]
                # A weight of exactly 0 never occurs here, so inf and NaN reach whoever sees them.
                out[at + t, h] = p @ vis
        at += n
    return out


# Groups around the 16-row tile, block sizes below, at and above the 16-key tile, token counts whose
# (token, head) rows end inside, at and just past a 16-row tile, and a context of several rounds. (One head
# per kv head runs the matrix-core kernel from 8 kv heads on here, the VALU kernel below.)
@pytest.mark.parametrize("d,hq,hkv,bs", [(64, 14, 2, 16), (64, 1, 1, 1), (64, 16, 1, 8), (64, 15, 1, 64), (128, 8, 2, 32),
                                         (128, 4, 4, 16), (64, 8, 8, 4), (128, 8, 8, 16), (64, 16, 8, 32)])
def test_prefill_tiles(gpu, d, hq, hkv, bs):
    from engine import paged_ops

    starts, lengths = [0, 130, 3, 0, 60], [1, 5, 33, 8, 2]
    announce(f"fp32 prefill d={d} hq={hq} hkv={hkv} bs={bs}")
    k, v, tab, gen = _pool(gpu, hkv, d, bs, [a + n for a, n in zip(starts, lengths)], seed=d + hq + bs)
    q = torch.randn(sum(lengths), hq, d, generator=gen, device=gpu)
    cu = torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()], dtype=torch.int32, device=gpu)
    st = torch.tensor(starts, dtype=torch.int32, device=gpu)
    got = paged_ops.paged_prefill(q, k, v, tab, cu, st, max(lengths))
    want = _exact(q, k, v, tab, starts, lengths, bs)
    # fp32 dot products of d terms and weighted sums of at most 135: their errors stay within
    # (d + 135) / 8 roundings of the largest value (independent signs, 8 deviations).
    bound = (d + 135) / 8 * 2.0 ** -24 * float(v.abs().max())
    assert float((got.double() - want).abs().max()) <= bound


@pytest.mark.parametrize("d,hq,hkv,bs", [(64, 14, 2, 16), (128, 16, 1, 8)])
def test_values_that_are_not_finite_reach_only_rows_that_see_them(gpu, d, hq, hkv, bs):
    """Several tokens share a row tile: an inf or NaN in a later token's value must not reach the earlier ones."""
    from engine import paged_ops

    announce(f"fp32 prefill with inf and NaN values d={d} hq={hq}")
    starts, lengths = [20, 0], [9, 17]
    k, v, tab, gen = _pool(gpu, hkv, d, bs, [29, 17], seed=5)

    def poke(seq, pos, dim, x):
        v[int(tab[seq, pos // bs]), :, pos % bs, dim] = x

    poke(0, 24, 3, float("inf"))
    poke(0, 27, 3, float("-inf"))
    poke(0, 26, d - 1, float("nan"))
    poke(1, 11, 17, float("inf"))
    q = torch.randn(26, hq, d, generator=gen, device=gpu)
    cu = torch.tensor([0, 9, 26], dtype=torch.int32, device=gpu)
    st = torch.tensor(starts, dtype=torch.int32, device=gpu)
    got = paged_ops.paged_prefill(q, k, v, tab, cu, st, 17).double()
    want = _exact(q, k, v, tab, starts, lengths, bs)
    fine = torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), fine)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got[~fine].nan_to_num(0.5), want[~fine].nan_to_num(0.5))
    assert float((got[fine] - want[fine]).abs().max()) <= 1e-5


def test_decode_agrees_with_the_valu_kernel(gpu):
    """Both fp32 decode kernels over lengths at tile, step and partition edges, group sizes 1 to 16."""
    from engine import _native, paged_ops

    lens = [1, 15, 16, 17, 127, 128, 129, 255, 256, 257, 1000, 0]
    for d, hq, hkv, bs in ((64, 14, 2, 16), (128, 16, 1, 4), (64, 3, 3, 32)):
        announce(f"fp32 decode d={d} hq={hq} hkv={hkv} bs={bs}")
        k, v, tab, gen = _pool(gpu, hkv, d, bs, lens, seed=d + bs)
        q = torch.randn(len(lens), hq, d, generator=gen, device=gpu)
        ctx = torch.tensor(lens, dtype=torch.int32, device=gpu)
        got = paged_ops.paged_decode(q, k, v, tab, ctx)
        prev = _native.set_decode_algo("valu")
        want = paged_ops.paged_decode(q, k, v, tab, ctx)
        _native.set_decode_algo(prev)
        # Each within d / 8 + sqrt(keys) roundings of the exact value.
        assert float((got - want).abs().max()) <= 2 * (d / 8 + 32) * 2.0 ** -24 * float(v.abs().max())
        assert not got[-1].any()
        # An unaligned q is read 4 bytes at a time.
        flat = torch.empty(q.numel() + 1, device=gpu)
        odd = flat[1:].view_as(q).copy_(q)
        assert torch.equal(paged_ops.paged_decode(odd, k, v, tab, ctx), got)


def _minus_infinity(k, tab, spans, bs):
    """Keys of sequence i at positions [a, b) score -inf for a query whose first element is positive."""
    for i, spans_i in enumerate(spans):
        for a, b in spans_i:
            for pos in range(a, b):
                k[int(tab[i, pos // bs]), :, pos % bs, 0] = -math.inf


@pytest.mark.parametrize("algo", ["auto", "valu"])
@pytest.mark.parametrize("d,hq,hkv,bs", [(64, 14, 2, 16), (128, 16, 2, 8), (64, 16, 1, 64), (32, 3, 3, 16), (256, 4, 2, 1)])
def test_a_score_of_minus_infinity_weighs_nothing(gpu, algo, d, hq, hkv, bs):
    """Whole tiles, wavefronts and partitions of keys that score -inf, before, between and after finite ones."""
    from engine import _native, paged_ops

    announce(f"fp32 scores of -inf d={d} hq={hq} bs={bs} {algo}")
    lens = [100, 300, 520, 17, 64]
    spans = [[(0, 64)], [(0, 256), (258, 300)], [(1, 519)], [(0, 16)], [(16, 64)]]
    k, v, tab, gen = _pool(gpu, hkv, d, bs, lens, seed=d + bs)
    _minus_infinity(k, tab, spans, bs)
    q = torch.randn(len(lens), hq, d, generator=gen, device=gpu)
    q[:, :, 0] = 1.0
    ctx = torch.tensor(lens, dtype=torch.int32, device=gpu)
    prev = _native.set_decode_algo(algo)
    got = paged_ops.paged_decode(q, k, v, tab, ctx)
    _native.set_decode_algo(prev)
    want = _exact(q, k, v, tab, [n - 1 for n in lens], [1] * len(lens), bs)
    # d / 8 + sqrt(keys) roundings of the largest value, as for the finite cases.
    bound = (d / 8 + 32) * 2.0 ** -24 * float(v.abs().max())
    assert float((got.double() - want).abs().max()) <= bound
    # The same keys under packed prefill: every row sees key 0, and the last ones more.
    starts, lengths = [40, 0], [60, 33]
    k, v, tab, gen = _pool(gpu, hkv, d, bs, [100, 33], seed=d)
    _minus_infinity(k, tab, [[(1, 97)], [(1, 20)]], bs)
    q = torch.randn(93, hq, d, generator=gen, device=gpu)
    q[:, :, 0] = 1.0
    cu = torch.tensor([0, 60, 93], dtype=torch.int32, device=gpu)
    st = torch.tensor(starts, dtype=torch.int32, device=gpu)
    got = paged_ops.paged_prefill(q, k, v, tab, cu, st, 60)
    want = _exact(q, k, v, tab, starts, lengths, bs)
    assert float((got.double() - want).abs().max()) <= bound


@pytest.mark.parametrize("d,bs", [(64, 16), (128, 8)])
@pytest.mark.parametrize("g", [1, 2, 3, 4, 6, 7, 8, 9, 15, 16])
def test_decode_of_every_group_size(gpu, d, bs, g):
    """The kernel that the group gets, and the matrix-core kernel where it is not that: one partition and several,
    whose merge splits a group of more than 8."""
    from engine import _native, paged_ops

    lens = [1, 16, 17, 255, 256, 257, 700, 0]
    k, v, tab, gen = _pool(gpu, 2, d, bs, lens, seed=d + g)
    q = torch.randn(len(lens), 2 * g, d, generator=gen, device=gpu)
    ctx = torch.tensor(lens, dtype=torch.int32, device=gpu)
    want = _exact(q[:-1], k, v, tab, [n - 1 for n in lens[:-1]], [1] * (len(lens) - 1), bs)
    for algo in ("auto", "mfma", "valu"):
        announce(f"fp32 decode d={d} group {g} {algo}")
        prev = _native.set_decode_algo(algo)
        got = paged_ops.paged_decode(q, k, v, tab, ctx)
        _native.set_decode_algo(prev)
        # d / 8 + sqrt(keys) roundings of the largest value.
        assert float((got[:-1].double() - want).abs().max()) <= (d / 8 + 32) * 2.0 ** -24 * float(v.abs().max())
        assert not got[-1].any()


# Single prompts of one kv head with the table as wide as the prompt: the last length that the VALU kernel gets and the
# first that the matrix-core kernel gets (h^2 keys > 16 d, h = heads per VALU workgroup), blocks of one key.
@pytest.mark.parametrize("d,g,first", [(64, 2, 257), (64, 4, 65), (64, 8, 17), (64, 9, 41), (128, 4, 129), (128, 7, 42),
                                       (128, 16, 33)])
def test_prefill_on_both_sides_of_the_rule(gpu, d, g, first):
    from engine import paged_ops

    for n in (first - 1, first):
        announce(f"fp32 prefill d={d} group {g} of {n} tokens")
        k, v, tab, gen = _pool(gpu, 1, d, 1, [n], seed=n)
        q = torch.randn(n, g, d, generator=gen, device=gpu)
        cu = torch.tensor([0, n], dtype=torch.int32, device=gpu)
        got = paged_ops.paged_prefill(q, k, v, tab, cu, cu[:1], n)
        want = _exact(q, k, v, tab, [0], [n], 1)
        # As in test_prefill_tiles, over at most 257 keys.
        assert float((got.double() - want).abs().max()) <= (d + 257) / 8 * 2.0 ** -24 * float(v.abs().max())
