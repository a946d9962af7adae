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
