"""The kernels that make a step's inputs: rotary tables, and a captured decode step's tables, slots and lengths."""

from __future__ import annotations

import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d,theta", [(64, 1e6), (128, 1e4), (2, 1e6), (6, 500.0)])
def test_rope_tables(gpu, dtype, d, theta):
    from engine.model import rope_cos_sin

    for shape in ((1, 1), (256, 1), (1, 1000), (3, 17)):
        announce(f"rope tables {dtype} d={d} theta={theta} {shape}")
        pos = torch.randint(0, 32768, shape, device=gpu)
        pos.view(-1)[0] = 0
        cos, sin = rope_cos_sin(pos, d, theta, dtype)
        half = d // 2
        assert cos.shape == sin.shape == (shape[0], 1, shape[1], d)
        assert torch.equal(cos[..., :half], cos[..., half:]) and torch.equal(sin[..., :half], sin[..., half:])
        inv = theta ** (-torch.arange(half, device=gpu, dtype=torch.float64) / half)
        ang = (pos.double().unsqueeze(-1) * inv).unsqueeze(1)
        # The angle is an fp32 product of a position and a frequency that itself took four fp32
        # roundings (exponent times log theta, pow within an ulp, reciprocal); cos and sin move by
        # at most the angle's error, and round to the dtype.
        u = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
        bound = ang.abs() * 2.0 ** -24 * (6 + 14) + 2.0 ** -22 + u
        assert ((cos[..., :half].double() - ang.cos()).abs() <= bound).all()
        assert ((sin[..., :half].double() - ang.sin()).abs() <= bound).all()
        # Positions the kernel does not take go through torch and give the same values to that bound.
        odd = torch.stack([pos, pos], dim=-1)[..., 0]
        c2, s2 = rope_cos_sin(odd, d, theta, dtype)
        assert ((c2.double() - cos.double()).abs()[..., :half] <= 2 * bound).all()
        assert ((s2.double() - sin.double()).abs()[..., :half] <= 2 * bound).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d", [2, 6, 48, 64, 80, 96, 112, 128, 160, 192])
def test_rope_tables_are_the_torch_steps_bit_for_bit(gpu, dtype, d):
    """Head sizes that are no power of two too, where a quotient by d and a product with 1 / d differ."""
    from engine.model import rope_cos_sin

    announce(f"rope tables against torch {dtype} d={d}")
    pos = torch.cat([torch.arange(2048, device=gpu), torch.randint(2048, 1 << 20, (512,), device=gpu)])[None]
    for theta in (1e6, 1e4, 10000.1, 3):
        cos, sin = rope_cos_sin(pos, d, theta, dtype)
        c2, s2 = rope_cos_sin(torch.stack([pos, pos], dim=-1)[..., 0], d, theta, dtype)  # strided: torch's own ops
        assert torch.equal(cos, c2) and torch.equal(sin, s2), theta


@pytest.mark.parametrize("bs", [1, 16, 64])
def test_decode_prepare(gpu, bs):
    from engine import paged_ops

    for batch, width, journal in ((1, 1, 0), (3, 7, 5), (40, 300, 64), (256, 513, 512)):
        announce(f"decode_prepare bs={bs} batch={batch} width={width} journal={journal}")
        gen = torch.Generator(device=gpu).manual_seed(batch + bs)
        n_rows = batch + 5
        rows = torch.randint(0, 1000, (n_rows, width), generator=gen, device=gpu, dtype=torch.int32)
        flat = torch.randperm(n_rows * width, generator=gen, device=gpu)[:min(journal, n_rows * width)].contiguous()
        block = torch.randint(0, 1 << 20, flat.shape, generator=gen, device=gpu)
        ids = torch.randperm(n_rows, generator=gen, device=gpu)[:batch].contiguous()
        pos = torch.randint(0, width * bs, (batch,), generator=gen, device=gpu)
        want = rows.clone().view(-1)
        want[flat] = block.to(torch.int32)
        want = want.view(n_rows, width)[ids]
        tables = torch.full((batch + 2, width), -1, dtype=torch.int32, device=gpu)
        slots = torch.zeros(batch, dtype=torch.int64, device=gpu)
        lens = torch.zeros(batch, dtype=torch.int32, device=gpu)
        paged_ops.decode_prepare(rows, flat, block, ids, pos, tables, width, slots, lens, bs)
        assert torch.equal(tables[:batch], want) and (tables[batch:] == -1).all()
        assert torch.equal(slots, want.gather(1, (pos // bs)[:, None])[:, 0].long() * bs + pos % bs)
        assert torch.equal(lens.long(), pos + 1)
