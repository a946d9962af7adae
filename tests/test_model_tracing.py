"""The model's modules under scripting, tracing and whole-graph compilation, on the CPU and on the GPU."""

from __future__ import annotations

import pytest
import torch

from conftest import HAS_GPU


def _check(dev):
    from engine.model import MLP, Qwen2Config, RMSNorm, rope_cos_sin

    cfg = Qwen2Config(vocab_size=64, hidden_size=64, intermediate_size=128, num_layers=1, num_heads=2, num_kv_heads=1,
                      head_dim=32)
    norm, mlp = RMSNorm(64, 1e-6).to(dev), MLP(cfg).to(dev)
    x = torch.randn(5, 64, device=dev)
    pos = torch.arange(5, device=dev)[None]

    def table(p):
        return rope_cos_sin(p, 32, 1e6, torch.float32)[0]

    with torch.no_grad():
        for mod in (norm, mlp):
            want = mod(x)
            for made in (torch.jit.script(mod), torch.jit.trace(mod, x),
                         torch.compile(mod, backend="eager", fullgraph=True)):
                torch.testing.assert_close(made(x), want, rtol=1e-5, atol=1e-6)
        torch.testing.assert_close(torch.compile(table, backend="eager", fullgraph=True)(pos), table(pos), rtol=1e-5,
                                   atol=1e-5)


def test_modules_can_be_scripted_traced_and_compiled():
    _check("cpu")


@pytest.mark.gpu
@pytest.mark.skipif(not HAS_GPU, reason="no ROCm GPU in this environment")
def test_modules_can_be_scripted_traced_and_compiled_on_the_gpu():
    _check("cuda")


def _check_symbolic(dev):
    """torch.fx: every module, and a model whose context is a constant, records the torch ops and gives their values."""
    from engine.model import MLP, DecoderLayer, Qwen2Config, Qwen2ForCausalLM, RMSNorm, rope_cos_sin

    cfg = Qwen2Config(vocab_size=64, hidden_size=64, intermediate_size=128, num_layers=2, num_heads=2, num_kv_heads=1,
                      head_dim=32)

    class Same:
        def attend(self, layer_idx, q, k, v):
            return q

    class OfConstant(torch.nn.Module):  # the weights are symbols, the input is not
        def __init__(self):
            super().__init__()
            self.norm, self.layer = RMSNorm(64, 1e-6), DecoderLayer(cfg, 0)
            self.x = torch.randn(1, 5, 64, device=dev)
            self.cos = torch.ones(1, 1, 5, 32, device=dev)

        def forward(self, y):
            return self.norm(self.x) + self.layer(self.x, self.cos, self.cos * 0, Same()) + y

    class Whole(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.model = Qwen2ForCausalLM(cfg)

        def forward(self, ids, pos):
            return self.model(ids, pos, Same())

    x = torch.randn(1, 5, 64, device=dev)
    pos = torch.arange(5, device=dev)[None]
    with torch.no_grad():
        for mod, args in ((RMSNorm(64, 1e-6), (x,)), (MLP(cfg), (x,)), (OfConstant(), (x,)), (Whole(), (pos, pos))):
            mod = mod.to(dev)
            made = torch.fx.symbolic_trace(mod)
            torch.testing.assert_close(made(*args), mod(*args), rtol=1e-5, atol=1e-5)
        made = torch.fx.symbolic_trace(rope_cos_sin, concrete_args={"head_dim": 32, "theta": 1e6, "dtype": torch.float32})
        for a, b in zip(made(pos, 32, 1e6, torch.float32), rope_cos_sin(pos, 32, 1e6, torch.float32)):
            torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5)


def test_modules_can_be_traced_symbolically():
    _check_symbolic("cpu")


@pytest.mark.gpu
@pytest.mark.skipif(not HAS_GPU, reason="no ROCm GPU in this environment")
def test_modules_can_be_traced_symbolically_on_the_gpu():
    _check_symbolic("cuda")


def test_a_default_device_is_no_observer_and_other_modes_are():
    """What the rule for the layer kernels takes for somebody watching the torch calls."""
    from engine import layer_ops
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Seen(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatched(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    assert not layer_ops._observed()
    with torch.device("cpu"):
        assert not layer_ops._observed()
        with torch.device("meta"):
            assert not layer_ops._observed()
            with Seen():
                assert layer_ops._observed()
        with Dispatched():
            assert layer_ops._observed()
    torch.set_default_device("cpu")
    try:
        assert not layer_ops._observed()
        with Seen():
            assert layer_ops._observed()
    finally:
        torch.set_default_device(None)


@pytest.mark.gpu
@pytest.mark.skipif(not HAS_GPU, reason="no ROCm GPU in this environment")
def test_layer_kernels_run_under_a_default_device(monkeypatch):
    from engine import layer_ops
    from engine.model import DecoderLayer, Qwen2Config, rope_cos_sin

    cfg = Qwen2Config(vocab_size=64, hidden_size=64, intermediate_size=128, num_layers=1, num_heads=2, num_kv_heads=1,
                      head_dim=32)

    class Same:
        def attend(self, layer_idx, q, k, v):
            return q

    layer = DecoderLayer(cfg, 0).to("cuda").requires_grad_(False)
    x, pos = torch.randn(2, 3, 64, device="cuda"), torch.arange(3, device="cuda").repeat(2, 1)
    calls = []
    tables = layer_ops.rope_tables
    monkeypatch.setattr(layer_ops, "rope_tables", lambda *a: calls.append(tables(*a)) or calls[-1])
    with torch.inference_mode():
        cos, sin = rope_cos_sin(pos, 32, 1e6, torch.float32)
        want = layer(x, cos, sin, Same())
        for dev in ("cuda", "cpu", "meta"):
            with torch.device(dev):
                assert layer._fusable(x)
                cos, sin = rope_cos_sin(pos, 32, 1e6, torch.float32)
                assert torch.equal(layer(x, cos, sin, Same()), want)
    assert len(calls) == 4 and all(c is not None for c in calls)
