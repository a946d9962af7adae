"""Which layers and operands the fused layer kernels and the step kernels may be given: the rest is refused on the host."""

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


def test_a_submodule_whose_call_means_something_else_is_called(monkeypatch):
    """Another forward, on the class or on the object, a hook or a compiled call: the fused steps pass none of them by."""
    from engine import layer_ops
    from engine.model import MLP, Attention, RMSNorm

    monkeypatch.setattr(layer_ops, "_open", lambda x: True)
    monkeypatch.setattr(layer_ops, "_operands", lambda x, *others: True)
    x = torch.zeros(8, 1, 64)
    for cls in (RMSNorm, Attention, MLP, nn.Linear):
        with monkeypatch.context() as m:
            m.setattr(cls, "forward", lambda self, *args: args[0])
            assert not _layer()._fusable(x)
    for change in (lambda m: setattr(m.mlp, "forward", lambda y: y), lambda m: m.attn.o_proj.compile(backend="eager"),
                   lambda m: m.input_norm.register_forward_pre_hook(lambda *a: None)):
        layer = _layer()
        assert layer._fusable(x)
        change(layer)
        assert not layer._fusable(x)


def _bad_calls():
    from engine import layer_ops as lo

    def z(*shape, dtype=torch.bfloat16):
        return torch.zeros(shape, dtype=dtype)

    x, w, n = z(8, 1, 64), z(96, 64), z(64)
    cs = z(8, 1, 1, 32)
    return [
        ("norm weight of another width", ValueError, lambda: lo.rms_norm(x, z(32), 1e-6)),
        ("norm weight with two dimensions", ValueError, lambda: lo.rms_norm(x, z(1, 64), 1e-6)),
        ("rows without elements", ValueError, lambda: lo.rms_norm(z(3, 0), z(0), 1e-6)),
        ("delta of fewer rows", ValueError, lambda: lo.add_rms_norm(x, z(1, 1, 64), n, 1e-6)),
        ("norm weight of another dtype", TypeError, lambda: lo.rms_norm(x, z(64, dtype=torch.float32), 1e-6)),
        ("a dtype without kernels", TypeError, lambda: lo.rms_norm(x.double(), n.double(), 1e-6)),
        ("strided rows", ValueError, lambda: lo.rms_norm(z(64, 8).t(), n, 1e-6)),
        ("odd gate_up", ValueError, lambda: lo.silu_mul(z(4, 33))),
        ("strided gate_up", ValueError, lambda: lo.silu_mul(z(4, 64)[:, :32])),
        ("rows twice the weight's width", ValueError, lambda: lo.norm_linear(x, z(32), 1e-6, z(96, 32))),
        ("norm of another width", ValueError, lambda: lo.norm_linear(x, z(32), 1e-6, w)),
        ("short bias", ValueError, lambda: lo.norm_linear(x, n, 1e-6, w, z(48))),
        ("bias beside gating", ValueError, lambda: lo.norm_linear(x, n, 1e-6, w, z(96), gate_up=True)),
        ("rows twice the weight's width", ValueError, lambda: lo.qkv_linear(x, None, 0.0, z(96, 32), None, cs, cs, 3)),
        ("tables of fewer rows", ValueError, lambda: lo.qkv_linear(x, n, 1e-6, w, None, cs[:1], cs[:1], 3)),
        ("sin unlike cos", ValueError, lambda: lo.qkv_linear(x, n, 1e-6, w, None, cs, z(8, 1, 1, 16), 3)),
        ("short bias", ValueError, lambda: lo.qkv_linear(x, n, 1e-6, w, z(64), cs, cs, 3)),
        ("tables of another dtype", TypeError, lambda: lo.qkv_linear(x, n, 1e-6, w, None, cs.float(), cs.float(), 3)),
        ("rows twice the weight's width", ValueError, lambda: lo.linear_residual(x, z(64, 32), x)),
        ("residual of fewer rows", ValueError, lambda: lo.linear_residual(x, z(64, 64), x[:4])),
        ("residual of another width", ValueError, lambda: lo.linear_residual(x, w, x)),
        ("host tensors", RuntimeError, lambda: lo.linear_residual(x, z(64, 64), x)),
        ("host tensors", RuntimeError, lambda: lo.silu_mul(z(4, 64))),
    ]


@pytest.mark.parametrize("i", range(23))
def test_the_functions_refuse_operands_their_kernels_cannot_read(monkeypatch, i):
    from engine import _native

    def load():
        raise AssertionError("a launch was reached")

    monkeypatch.setattr(_native, "load", load)
    calls = _bad_calls()
    assert len(calls) == 23
    what, error, call = calls[i]
    with pytest.raises(error):
        call()


@pytest.mark.parametrize("change", [
    {"cu_q": [0, 3]}, {"cu_q": [[0, 3, 5]]}, {"cu_q": [0, 3, 5, 6]}, {"ctx_start": [[0, 0]]}, {"block_tables": [[0, 1]]},
    {"block_tables": [0, 1]}, {"dtype": torch.int64}, {"strided": True}, {"n_tokens": -1}, {"max_q_len": -3},
])
def test_prefill_index_refuses_tensors_that_do_not_match(monkeypatch, change):
    """cu_q holds one entry more than there are sequences, and every sequence has a table row."""
    from engine import _native, paged_ops

    def load():
        raise AssertionError("a launch was reached")

    monkeypatch.setattr(_native, "load", load)
    dt = change.get("dtype", torch.int32)
    cu, start, tab = (torch.tensor(change.get(n, d), dtype=dt) for n, d in (
        ("cu_q", [0, 3, 5]), ("ctx_start", [0, 0]), ("block_tables", [[0, 1], [2, 3]])))
    if change.get("strided"):
        tab = tab.t()
    with pytest.raises(ValueError):
        paged_ops.prefill_index(cu, start, tab, change.get("n_tokens", 5), change.get("max_q_len", 3), 4)


def test_a_kept_step_serves_only_layers_that_both_pools_hold():
    """Later calls add the layer's offset to the pools' addresses: a layer that one of them lacks is checked in full."""
    from engine import _native, paged_ops

    calls = paged_ops._LayerCalls()
    k, v = torch.zeros(4, 3, 2, 16, 8), torch.zeros(2, 3, 2, 16, 8)
    calls._keep("decode", ("key",), _native.DecodeStep(), k, v, ())
    assert calls._hit("decode", ("key",), 1) is not None
    for layer in (2, 3, 4, -1, True, 1.0):
        assert calls._hit("decode", ("key",), layer) is None


@pytest.mark.parametrize("rule,rows,n,k,pays", [
    ("norm_linear_pays", 8, 1152, 896, True), ("norm_linear_pays", 256, 1152, 896, True),
    ("norm_linear_pays", 257, 1152, 896, False), ("norm_linear_pays", 16, 2048, 4096, True),
    ("norm_linear_pays", 8, 4608, 3584, False), ("norm_linear_pays", 32, 1024, 4096, True),
    ("norm_linear_pays", 33, 1024, 4096, False), ("norm_linear_pays", 64, 2048, 2048, True),
    ("norm_linear_pays", 65, 3072, 1344, False), ("norm_linear_pays", 129, 1024, 1536, False),
    ("norm_linear_pays", 8, 1160, 896, False), ("norm_linear_pays", 8, 1152, 900, False),
    ("norm_gate_up_pays", 16, 22016, 2048, True), ("norm_gate_up_pays", 1, 16384, 3072, False),
    ("norm_gate_up_pays", 64, 9728, 896, True), ("norm_gate_up_pays", 65, 9728, 896, False),
    ("norm_gate_up_pays", 17, 12288, 1024, False), ("norm_gate_up_pays", 64, 12288, 1024, True),
    ("norm_gate_up_pays", 33, 8192, 1536, False), ("linear_residual_pays", 16, 3584, 18944, True),
    ("linear_residual_pays", 1, 5120, 14336, False), ("linear_residual_pays", 64, 896, 4864, True),
    ("linear_residual_pays", 65, 896, 4864, False), ("linear_residual_pays", 33, 2048, 2560, False),
    ("linear_residual_pays", 32, 1536, 1536, True), ("linear_residual_pays", 33, 1536, 1536, False),
    ("linear_residual_pays", 256, 896, 896, True), ("linear_residual_pays", 256, 512, 2048, False),
])
def test_the_rules_take_the_shapes_that_were_measured_faster(rule, rows, n, k, pays):
    from engine import layer_ops

    for dtype in (torch.float16, torch.bfloat16):
        assert getattr(layer_ops, rule)(rows, torch.empty(n, k, dtype=dtype, device="meta")) is pays
    assert not getattr(layer_ops, rule)(rows, torch.empty(n, k, device="meta"))


@pytest.mark.gpu
@torch.inference_mode()
def test_a_layer_whose_widths_disagree_raises_on_the_gpu_as_anywhere(gpu):
    """torch's shape errors, before anything of the layer's own is launched out of range; a bias row broadcasts."""
    class Same:
        def attend(self, layer_idx, q, k, v):
            return q

    dt = torch.bfloat16
    x = torch.randn(8, 1, 64, device=gpu).to(dt)
    cs = torch.ones(8, 1, 1, 16, device=gpu, dtype=dt)

    def run(change):
        torch.manual_seed(0)
        layer = _layer()
        change(layer)
        layer = layer.to(gpu, dt)
        return layer._fusable(x), layer(x, cs, cs * 0, Same())

    for bad in (lambda m: _resized(m.attn.o_proj, 64, 32), lambda m: _resized(m.attn.o_proj, 32, 64),
                lambda m: _resized(m.attn.qkv_proj, 128, 64, bias=64), lambda m: _resized(m.mlp.down_proj, 64, 64)):
        with pytest.raises(RuntimeError):
            run(bad)
    fused, want = run(lambda m: None)
    assert fused

    def row(m):
        m.attn.qkv_proj.bias = nn.Parameter(m.attn.qkv_proj.bias[None], requires_grad=False)

    fused, got = run(row)
    assert not fused
    # The same layer through torch's ops: each side rounds every intermediate once or twice.
    assert float((got.double() - want.double()).norm() / want.double().norm()) <= 8 * 2.0 ** -8
