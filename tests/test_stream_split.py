"""How many pieces the decode split can cut a segment into, and the launches that follow from it."""

from __future__ import annotations

import random

import pytest
import torch

from conftest import announce


def test_a_segment_of_n_tiles_meets_at_most_half_of_them_plus_one_ranges():
    """The bound by which a call with short tables skips the merge's fold: W <= ceil(T / 4) ranges of T tiles
    (fewer where the grid or the piece cap is smaller), range g = [g T / W, (g + 1) T / W)."""
    rng = random.Random(1)
    sizes = [1, 2, 3, 4, 5, 7, 9, 15, 16, 17, 30, 61, 62, 63, 64]
    for _ in range(40000):
        segs = [rng.choice(sizes) for _ in range(rng.randint(1, 8))]
        total = sum(segs)
        w = -(-total // 4)
        if rng.random() < 0.3:
            w = rng.randint(1, w)
        s0 = 0
        for n in segs:
            pieces = ((s0 + n) * w - 1) // total - ((s0 + 1) * w - 1) // total + 1
            assert pieces <= n // 2 + 1, (segs, n, w)
            s0 += n


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_short_tables_give_the_same_bits_with_and_without_the_fold(gpu, dtype):
    """Tables of 62 tiles run no fold, wider tables of the same sequences do: the same split, the same sums."""
    from engine import paged_ops

    announce(f"decode with and without the fold, {dtype}")
    gen = torch.Generator(device=gpu).manual_seed(3)
    for batch, hkv, hq, d, bs in ((1, 2, 14, 64, 16), (4, 4, 28, 128, 32), (8, 2, 14, 64, 64)):
        lens = [max(1, 992 - 61 * i) for i in range(batch)]
        need = -(-992 // bs)
        k = torch.randn(batch * need, hkv, bs, d, generator=gen, device=gpu).to(dtype)
        v = torch.randn(batch * need, hkv, bs, d, generator=gen, device=gpu).to(dtype)
        q = torch.randn(batch, hq, d, generator=gen, device=gpu).to(dtype)
        narrow = torch.randperm(batch * need, generator=gen, device=gpu).to(torch.int32).view(batch, need)
        wide = torch.full((batch, 2 * need), -1, dtype=torch.int32, device=gpu)
        wide[:, :need] = narrow
        ctx = torch.tensor(lens, dtype=torch.int32, device=gpu)
        for planned in (False, True):
            outs = []
            for bt in (narrow, wide):
                plan = paged_ops.decode_plan(ctx, bt, hq, hkv, d, bs, dtype) if planned else None
                outs.append(paged_ops.paged_decode(q, k, v, bt, ctx, plan=plan))
            assert torch.equal(outs[0], outs[1]), (batch, planned)
