"""Lifetimes around graph capture: no reference cycle keeps a decoder, and no collection runs while a stream records."""

from __future__ import annotations

import gc
import threading
import types
import weakref

import pytest
import torch


def test_no_collection_while_any_thread_is_inside():
    from engine.cuda_graphs import _NoCollection

    guard, inside, leave, seen = _NoCollection(), threading.Event(), threading.Event(), []

    def other():
        with guard:
            inside.set()
            leave.wait(10)

    assert gc.isenabled()
    t = threading.Thread(target=other)
    with guard:
        t.start()
        assert inside.wait(10)
        assert not gc.isenabled()
        with guard:
            seen.append(gc.isenabled())
        seen.append(gc.isenabled())
    seen.append(gc.isenabled())  # the other thread is still inside
    leave.set()
    t.join(10)
    assert seen == [False] * 3 and gc.isenabled()
    with pytest.raises(KeyError):
        with guard:
            raise KeyError
    assert gc.isenabled()
    gc.disable()
    try:
        with guard:
            pass
        assert not gc.isenabled()  # left as it was found
    finally:
        gc.enable()


def test_a_context_holds_what_its_graph_reads_and_not_its_decoder(monkeypatch):
    from engine import cuda_graphs

    class Owner(types.SimpleNamespace):
        pass

    monkeypatch.setattr(cuda_graphs.paged_ops, "prepare_decode_plan", lambda *a, **k: (None, None))
    cache = types.SimpleNamespace(block_size=16, head_dim=8, num_kv_heads=1, k=torch.zeros(1))
    model = Owner(cfg=types.SimpleNamespace(num_heads=2))
    inputs, rows = torch.zeros(16), Owner()
    owner = Owner(cache=cache, model=model, fuse_rope=True, device_tables=rows, _inputs=inputs, positions=inputs[:4],
                  tables=torch.zeros(4, 2), slot_mapping=torch.zeros(4), context_lens=torch.zeros(4),
                  workspace=torch.zeros(8))
    ctx = cuda_graphs._GraphDecodeContext(owner, 2, 32)
    assert ctx.owner is owner
    refs = [weakref.ref(x) for x in (model, rows)]
    gone, ws = weakref.ref(owner), owner.workspace.data_ptr()
    del owner, model, rows
    assert gone() is None and all(r() is not None for r in refs) and ctx.workspace.data_ptr() == ws
    with pytest.raises(ReferenceError):
        ctx.owner


@pytest.mark.gpu
@torch.inference_mode()
def test_a_dropped_decoder_goes_at_once_and_the_next_is_recorded_without_collections(gpu):
    from engine.cuda_graphs import GraphedDecoder
    from engine.kv_cache import PagedKVCache
    from engine.model import Qwen2Config, Qwen2ForCausalLM

    cfg = Qwen2Config(vocab_size=64, hidden_size=128, intermediate_size=256, num_layers=2, num_heads=2, num_kv_heads=1,
                      head_dim=64)
    model = Qwen2ForCausalLM(cfg).to(gpu, torch.bfloat16).requires_grad_(False)
    enabled, logits = [], []
    model.layers[0].register_forward_hook(lambda *a: enabled.append(gc.isenabled()))
    for _ in range(3):
        cache = PagedKVCache(2, 1, 64, num_blocks=32, block_size=16, max_seqs=4, max_len=128, dtype=torch.bfloat16,
                             device=gpu)
        slots = [cache.allocate(20) for _ in range(3)]
        cache.k.fill_(0.25)
        cache.v.fill_(0.5)
        for s in slots:
            cache.lengths[s] = 11
        decoder = GraphedDecoder(model, cache, max_batch=4)
        decoder.capture()
        logits.append(decoder.decode(slots, [1, 2, 3]).clone())
        gone = weakref.ref(decoder)
        del decoder
        assert gone() is None
    assert enabled and not any(enabled) and gc.isenabled()
    assert all(torch.equal(x, logits[0]) for x in logits)
