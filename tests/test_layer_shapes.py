"""Which layers and operands the fused layer kernels may be given: everything else is refused before a launch."""

from __future__ import annotations

import pytest
import torch
from torch import nn


def _layer(hidden=64, inter=128, heads=4, kv=2, d=16):
    from engine.model import DecoderLayer, Qwen2Config

    cfg = Qwen2Config(vocab_size=64, hidden_size=hidden, intermediate_size=inter, num_layers=1, num_heads=heads,
                      num_kv_heads=kv, head_dim=d)
    return DecoderLayer(cfg, 0).requires_grad_(False)


def _resized(linear, out, inp, bias=None):
    """The module as it is, with weights of another shape (what a pruned or wrongly loaded checkpoint leaves)."""
    linear.weight = nn.Parameter(torch.zeros(out, inp), requires_grad=False)
    if bias is not None:
        linear.bias = nn.Parameter(torch.zeros(bias), requires_grad=False)


@pytest.mark.parametrize("wrong", [
    lambda m: _resized(m.attn.o_proj, 64, 32),  # 8 rows of 64 would be read as 16 of 32
    lambda m: _resized(m.attn.o_proj, 32, 64),
    lambda m: _resized(m.attn.qkv_proj, 128, 64, bias=64),
    lambda m: _resized(m.attn.qkv_proj, 128, 64, bias=(1, 128)),
    lambda m: _resized(m.attn.qkv_proj, 144, 64, bias=144),
    lambda m: _resized(m.attn.qkv_proj, 128, 32),
    lambda m: _resized(m.mlp.gate_up_proj, 256, 32),
    lambda m: _resized(m.mlp.gate_up_proj, 257, 64),
    lambda m: _resized(m.mlp.down_proj, 64, 64),
    lambda m: _resized(m.mlp.down_proj, 32, 128),
])
def test_a_layer_whose_widths_disagree_is_left_to_torch(monkeypatch, wrong):
    """torch's own products raise for such a layer (or broadcast its bias); the fused steps would run out of range."""
    from engine import layer_ops

    monkeypatch.setattr(layer_ops, "_open", lambda x: True)  # as for device tensors
    monkeypatch.setattr(layer_ops, "_operands", lambda x, *others: True)
    x = torch.zeros(8, 1, 64)
    layer = _layer()
    assert layer._fusable(x)
    wrong(layer)
    assert not layer._fusable(x)
