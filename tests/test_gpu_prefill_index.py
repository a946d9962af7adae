"""The index arrays of a packed prefill step against the host's own construction of them."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import announce

pytestmark = pytest.mark.gpu


# Lengths of nothing, one token, and around the 256 tokens of a workgroup; block sizes from one
# token to more than any sequence.
@pytest.mark.parametrize("block", [1, 16, 8192])
def test_prefill_context_indices(gpu, block):
    from engine.kv_cache import PagedKVCache

    lengths = [[1], [256, 0, 257, 1, 255], [3, 700], [0], [16] * 40]
    for n, lens in enumerate(lengths):
        starts = [(7 * i + n) % 40 for i in range(len(lens))]
        announce(f"prefill index block {block} lengths {lens[:6]}")
        cache = PagedKVCache(1, 1, 8, max(64, 4096 // block), block, max_seqs=64, max_len=16384, dtype=torch.float32,
                             device=gpu)
        # Blocks handed out in turns, so that tables are not runs of consecutive ids.
        slots = [cache.allocate(0) for _ in lens]
        for t in range(1, max(a + m for a, m in zip(starts, lens)) + 1):
            for s, a, m in zip(slots, starts, lens):
                if t <= a + m:
                    assert cache.ensure_capacity(s, t)
        for s, a in zip(slots, starts):
            cache.lengths[s] = a
        ctx = cache.packed_prefill_context(slots, lens)
        blocks, offsets = cache._write_index_np(slots, starts, lens)
        pos = np.concatenate([np.arange(a, a + m) for a, m in zip(starts, lens)])
        assert ctx.positions.dtype == ctx.slot_mapping.dtype == ctx.last_index.dtype == torch.int64
        assert ctx.positions.tolist() == pos.tolist()
        assert ctx.slot_mapping.tolist() == (blocks * block + offsets).tolist()
        assert ctx.last_index.tolist() == (np.cumsum(lens) - 1).tolist()
        assert [x.tolist() for x in ctx.write_at] == [blocks.tolist(), offsets.tolist()]
        assert ctx.cu_q.tolist() == [0, *np.cumsum(lens).tolist()] and ctx.ctx_start.tolist() == starts
        for row, s, a, m in zip(ctx.block_tables.tolist(), slots, starts, lens):
            table = cache.block_tables[s][:len(row)]
            assert row == table + [0] * (len(row) - len(table))


def test_prefill_context_is_ready_on_any_stream(gpu):
    """What the constructor made is in place when it returns, also for a stream that it did not run on."""
    from engine.kv_cache import PagedKVCache

    announce("prefill index: used on another stream")
    cache = PagedKVCache(1, 1, 8, 512, 16, max_seqs=8, max_len=4096, dtype=torch.float32, device=gpu)
    other = torch.cuda.Stream()
    busy = torch.randn(2048, 2048, device=gpu)
    for _ in range(5):
        slots = [cache.allocate(0) for _ in range(4)]
        for _ in range(20):
            busy = busy @ busy * 1e-3  # the constructor's stream has work queued before it
        ctx = cache.packed_prefill_context(slots, [300, 20, 1000, 5])
        with torch.cuda.stream(other):
            got = ctx.slot_mapping.clone(), ctx.positions.clone()
        other.synchronize()
        blocks, offsets = cache._write_index_np(slots, [0] * 4, [300, 20, 1000, 5])
        assert got[0].tolist() == (blocks * 16 + offsets).tolist()
        assert got[1].tolist() == [*range(300), *range(20), *range(1000), *range(5)]
        for s in slots:
            cache.free(s)


def test_prefill_context_needs_a_sequence(gpu):
    from engine.kv_cache import PagedKVCache

    cache = PagedKVCache(1, 1, 8, 8, 16, max_seqs=2, max_len=64, dtype=torch.float32, device=gpu)
    with pytest.raises(ValueError):
        cache.packed_prefill_context([], [])
