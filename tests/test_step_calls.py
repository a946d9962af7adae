"""What the layer calls of a step hold on to, and what a packed prefill's calls are bound to."""

from __future__ import annotations

import gc

import pytest
import torch
from torch.multiprocessing.reductions import StorageWeakRef


class _Library:
    """Takes every launch; a step struct's slot list is noted."""

    def __init__(self):
        self.slots = []

    def mip_paged_decode_workspace(self, *args):
        return 0

    def mip_prefill_step_append(self, step, *args):
        from engine import _native

        self.slots.append(_native.PrefillStep.from_address(step).slot_mapping)
        return 0

    def mip_kv_append(self, *args):
        self.slots.append(args[9])
        return 0

    def __getattr__(self, name):
        return lambda *args: 0


@pytest.fixture
def library(monkeypatch):
    """The native library replaced, so that calls on host tensors get as far as their launch."""
    from engine import _native, paged_ops

    lib = _Library()
    monkeypatch.setattr(_native, "load", lambda *a: lib)
    monkeypatch.setattr(paged_ops, "_require_device", lambda *tensors: None)
    monkeypatch.setattr(paged_ops, "_stream_ptr", lambda device: 0)
    return lib


def _qkv(rows, tokens, hq=4, hkv=2, d=16):
    return [torch.randn(rows, h, tokens, d) for h in (hq, hkv, hkv)]


@pytest.mark.parametrize("kind", ["prefill", "decode"])
def test_a_step_holds_none_of_its_layers_tensors(library, kind):
    """The first call of a kind lays out what the layers share; its q, k, v, tables of cos and sin, and output go free."""
    from engine import paged_ops

    k_pool, v_pool = torch.zeros(3, 9, 2, 16, 16), torch.zeros(3, 9, 2, 16, 16)
    tables = torch.arange(4, dtype=torch.int32).view(2, 2)
    lens = torch.tensor([5, 3], dtype=torch.int32)
    if kind == "prefill":
        slots = torch.arange(8)
        calls = paged_ops.PrefillStepCalls(tables, torch.tensor([0, 5, 8], dtype=torch.int32), lens * 0, slots, 5, 0.25)
        rows, tokens, cs = 1, 8, torch.ones(1, 1, 8, 16)
    else:
        slots = torch.arange(2)
        calls = paged_ops.DecodeStepCalls(tables, lens, slots, 0.25, 2, lambda heads, dtype: None)
        rows, tokens, cs = 2, 1, torch.ones(2, 1, 1, 16)
    seen = []
    for layer in range(2):
        q, k, v = _qkv(rows, tokens)
        cos, sin = cs.clone(), cs.clone()
        calls.rope_append(layer, q, k, v, cos, sin, k_pool, v_pool)
        if kind == "prefill":
            calls.append(layer, k, v, k_pool, v_pool)
        else:
            seen.append(StorageWeakRef(calls.append_attend(layer, q, k, v, k_pool, v_pool).untyped_storage()))
        out = calls.attend(layer, q, k_pool, v_pool)
        seen += [StorageWeakRef(t.untyped_storage()) for t in (q, k, v, cos, sin, out)]
    assert len(calls._cached) == 3
    assert not seen[-1].expired()
    del q, k, v, cos, sin, out
    gc.collect()
    assert all(r.expired() for r in seen)


def test_a_prefill_context_follows_what_is_assigned_to_it(library):
    """slot_mapping, the tables and write_at may be replaced between layers, as plain attributes may."""
    from engine.kv_cache import PagedKVCache

    cache = PagedKVCache(2, 2, 16, 32, 16, max_seqs=4, max_len=128, dtype=torch.float32, device="cpu")
    slots = [cache.allocate(0) for _ in range(2)]
    ctx = cache.packed_prefill_context(slots, [5, 20])
    _, k, v = _qkv(1, 25)
    blocks, offsets = ctx.write_at
    assert torch.equal(blocks * 16 + offsets, ctx.slot_mapping)
    for layer in range(2):
        ctx.calls.append(layer, k, v, cache.k, cache.v)
    first = ctx.slot_mapping
    ctx.slot_mapping = first.flip(0).contiguous()
    for layer in range(2):
        ctx.calls.append(layer, k, v, cache.k, cache.v)
    assert library.slots == [first.data_ptr()] * 2 + [ctx.slot_mapping.data_ptr()] * 2
    kept = ctx.calls
    ctx.other = 1
    assert ctx.calls is kept
    for name in ("block_tables", "cu_q", "ctx_start"):
        setattr(ctx, name, getattr(ctx, name).clone())
        assert ctx.calls is not kept and getattr(ctx.calls, name) is getattr(ctx, name)
        kept = ctx.calls
    ctx.write_at = (offsets, blocks)
    assert ctx.write_at[0] is offsets and ctx.write_at[1] is blocks
