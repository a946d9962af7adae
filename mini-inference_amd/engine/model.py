"""Qwen2 decoder used as the harness around the paged KV-cache kernels.

The attention layer hands its post-RoPE q, k, v to an ``AttentionContext`` and gets the
attention output back, exactly as engine/model.py:241-251 of the reference does
(``out = ctx.attend(self.layer_idx, q, k, v)``). The cache contexts in
:mod:`engine.kv_cache` implement that protocol with the HIP kernels; this module only
supplies the surrounding projections, norms, RoPE and MLP so that a full decode step can be
timed with random-init weights (no checkpoint is loaded). Norms, residual adds and the MLP's
gating run as fused kernels (:mod:`engine.layer_ops`) in inference on the GPU and as torch ops
everywhere else.

Shapes (reference engine/model.py:89-98): q ``[B, Hq, T, D]``, k and v
``[B, Hkv, T, D]``; ``attend`` returns ``[B, Hq, T, D]``.
"""

from __future__ import annotations

import math
from dataclasses import dataclass
from typing import Protocol

import torch
import torch.nn.functional as F
from torch import nn

from . import layer_ops


@dataclass(frozen=True)
class Qwen2Config:
    """Architecture numbers (field names as engine/model.py:37-86)."""

    vocab_size: int
    hidden_size: int
    intermediate_size: int
    num_layers: int
    num_heads: int
    num_kv_heads: int
    head_dim: int
    rms_norm_eps: float = 1e-6
    rope_theta: float = 1_000_000.0
    max_position_embeddings: int = 32768
    tie_word_embeddings: bool = True
    attention_bias: bool = True

    @property
    def q_size(self) -> int:
        return self.num_heads * self.head_dim

    @property
    def kv_size(self) -> int:
        return self.num_kv_heads * self.head_dim

    @classmethod
    def qwen2_5_0_5b(cls) -> "Qwen2Config":
        """Qwen2.5-0.5B: 24 layers, hidden 896, 14 query / 2 KV heads of 64, tied embeddings."""
        return cls(vocab_size=151936, hidden_size=896, intermediate_size=4864, num_layers=24, num_heads=14,
                   num_kv_heads=2, head_dim=64)

    @classmethod
    def qwen2_7b_like(cls) -> "Qwen2Config":
        """The 7B-class GQA shape: 28 layers, 28 query / 4 KV heads of 128."""
        return cls(vocab_size=152064, hidden_size=3584, intermediate_size=18944, num_layers=28, num_heads=28,
                   num_kv_heads=4, head_dim=128, tie_word_embeddings=False)


class AttentionContext(Protocol):
    """Receives one layer's post-RoPE q, k, v; stores k/v; returns attention output.

    A context whose ``fuse_rope`` attribute is true instead receives q and k before the
    rotary embedding, with the step's cos/sin tables, through
    ``attend_rope(layer_idx, q, k, v, cos, sin)``, and applies the rotation itself. One whose
    ``takes_rotated`` attribute is true as well may be given rotated q and k through ``attend``
    instead, where the layer has a cheaper place for the rotation (the end of its projection).
    """

    def attend(self, layer_idx: int, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor: ...


def _plain(module: nn.Module, cls: type) -> bool:
    """Whether calling ``module`` does what this file's (or torch's) ``cls.forward`` says and nothing else: its exact
    class, unpatched, uncompiled, no hooks.

    A fused step that passes a submodule's call by is only taken where nobody watches that call.
    """
    if torch.compiler.is_compiling():
        return False
    g = nn.modules.module
    return (type(module) is cls and cls.forward is _FORWARD[cls] and "forward" not in module.__dict__
            and module._compiled_call_impl is None and not module._forward_hooks
            and not module._forward_pre_hooks and not module._backward_hooks and not module._backward_pre_hooks
            and not g._global_forward_hooks and not g._global_forward_pre_hooks and not g._global_backward_hooks
            and not g._global_backward_pre_hooks)


class RMSNorm(nn.Module):
    """x / rms(x) * weight with the statistic taken in fp32, result cast back first."""

    def __init__(self, dim: int, eps: float) -> None:
        super().__init__()
        self.weight = nn.Parameter(torch.ones(dim))
        self.eps = eps

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if not torch.jit.is_scripting():
            if layer_ops.norm_usable(self.weight, x):
                return layer_ops._rms_norm(x, self.weight, self.eps)
        xf = x.float()
        inv = torch.rsqrt(xf.square().mean(dim=-1, keepdim=True) + self.eps)
        return self.weight * (xf * inv).to(x.dtype)


def rope_cos_sin(positions: torch.Tensor, head_dim: int, theta: float, dtype: torch.dtype):
    """cos/sin ``[B, 1, T, D]`` for per-token ``positions [B, T]`` (half-rotation layout)."""
    if not torch.jit.is_scripting():
        tables = layer_ops.rope_tables(positions, head_dim, theta, dtype)
        if tables is not None:
            return tables
    half = head_dim // 2
    inv_freq = 1.0 / (theta ** (torch.arange(half, device=positions.device, dtype=torch.float32) * 2.0 / head_dim))
    ang = positions.to(torch.float32).unsqueeze(-1) * inv_freq  # [B, T, D/2]
    ang = torch.cat((ang, ang), dim=-1).unsqueeze(1)
    return ang.cos().to(dtype), ang.sin().to(dtype)


def apply_rope(q: torch.Tensor, k: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor):
    def rot(x: torch.Tensor) -> torch.Tensor:
        a, b = x.chunk(2, dim=-1)
        return torch.cat((-b, a), dim=-1)

    return q * cos + rot(q) * sin, k * cos + rot(k) * sin


class Attention(nn.Module):
    def __init__(self, cfg: Qwen2Config, layer_idx: int) -> None:
        super().__init__()
        self.layer_idx = layer_idx
        self.cfg = cfg
        self.qkv_proj = nn.Linear(cfg.hidden_size, cfg.q_size + 2 * cfg.kv_size, bias=cfg.attention_bias)
        self.o_proj = nn.Linear(cfg.q_size, cfg.hidden_size, bias=False)

    def forward(self, x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, ctx: AttentionContext) -> torch.Tensor:
        return self.o_proj(self.attend(self.qkv_proj(x), cos, sin, ctx))

    def attend(self, qkv: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, ctx: AttentionContext,
               rotated: bool = False) -> torch.Tensor:
        """The part between the projections: ``[B, T, q + 2 kv]`` in, ``[B, T, q]`` out. ``rotated``: the rotary
        embedding has been applied."""
        c = self.cfg
        bsz, t, _ = qkv.shape
        q, k, v = qkv.split([c.q_size, c.kv_size, c.kv_size], dim=-1)
        q = q.view(bsz, t, c.num_heads, c.head_dim).transpose(1, 2)
        k = k.view(bsz, t, c.num_kv_heads, c.head_dim).transpose(1, 2)
        v = v.view(bsz, t, c.num_kv_heads, c.head_dim).transpose(1, 2)
        if rotated:
            out = ctx.attend(self.layer_idx, q, k, v)
        elif getattr(ctx, "fuse_rope", False):
            # The context rotates q and k itself (in place), fused with its KV append.
            out = ctx.attend_rope(self.layer_idx, q, k, v, cos, sin)
        else:
            q, k = apply_rope(q, k, cos, sin)
            out = ctx.attend(self.layer_idx, q, k, v)  # the call site the cache contexts serve
        return out.transpose(1, 2).reshape(bsz, t, c.q_size)


class MLP(nn.Module):
    def __init__(self, cfg: Qwen2Config) -> None:
        super().__init__()
        self.gate_up_proj = nn.Linear(cfg.hidden_size, 2 * cfg.intermediate_size, bias=False)
        self.down_proj = nn.Linear(cfg.intermediate_size, cfg.hidden_size, bias=False)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return self.down_proj(self.gated(self.gate_up_proj(x)))

    def gated(self, gate_up: torch.Tensor) -> torch.Tensor:
        if not torch.jit.is_scripting():
            if layer_ops.silu_mul_usable(gate_up):
                return layer_ops._silu_mul(gate_up)
        gate, up = gate_up.chunk(2, dim=-1)
        return F.silu(gate) * up


class DecoderLayer(nn.Module):
    def __init__(self, cfg: Qwen2Config, layer_idx: int) -> None:
        super().__init__()
        self.input_norm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)
        self.attn = Attention(cfg, layer_idx)
        self.post_attn_norm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)
        self.mlp = MLP(cfg)

    def forward(self, x, cos, sin, ctx):
        if self._fusable(x):
            x, delta = self._fused(x, None, cos, sin, ctx)
            return x if delta is None else x + delta
        x = x + self.attn(self.input_norm(x), cos, sin, ctx)
        return x + self.mlp(self.post_attn_norm(x))

    def _fusable(self, x: torch.Tensor) -> bool:
        """Whether the layer may run as its fused steps: unwatched submodules, operands the kernels take."""
        if not layer_ops._open(x):
            return False
        a, m, n1, n2 = self.attn, self.mlp, self.input_norm, self.post_attn_norm
        if not (_plain(n1, RMSNorm) and _plain(n2, RMSNorm) and _plain(a, Attention) and _plain(m, MLP)):
            return False
        linears = (a.qkv_proj, a.o_proj, m.gate_up_proj, m.down_proj)
        if not all(_plain(p, nn.Linear) for p in linears) or any(p.bias is not None for p in linears[1:]):
            return False
        w, bias, c = [p.weight for p in linears], a.qkv_proj.bias, a.cfg
        h, qkv, inter = x.shape[-1], c.q_size + 2 * c.kv_size, w[2].shape[0] // 2
        # Every width: the kernels take a shape that torch would refuse for a longer list of rows.
        return (x.dim() == 3 and w[0].shape == (qkv, h) and w[1].shape == (h, c.q_size) and w[2].shape == (2 * inter, h)
                and w[3].shape == (h, inter) and (bias is None or bias.shape == (qkv,))
                and n2.weight.shape == n1.weight.shape and layer_ops._norm_fits(n1.weight, x)
                and layer_ops._operands(x, n1.weight, n2.weight, *w, *(() if bias is None else (bias,))))

    def _fused(self, x, delta, cos, sin, ctx):
        """``forward`` of ``x + delta`` (None: of x), as ``(y, delta)`` whose sum it is (None: y is).

        Norms, bias, residual adds and gating run inside the linear layers where rows are few, and
        as one kernel each between library products where they are many; there the last residual
        add is left to the caller, which may have a norm to fuse it with.
        """
        a, m, n1, n2 = self.attn, self.mlp, self.input_norm, self.post_attn_norm
        rows = x.shape[0] * x.shape[1]
        w, c = a.qkv_proj.weight, a.cfg
        normed = None
        if delta is not None:
            x, normed = layer_ops._add_rms_norm(x, delta, n1.weight, n1.eps)
        # A context that takes rotated q and k in its fused append gets them from the projection itself.
        rotated = (getattr(ctx, "fuse_rope", False) and getattr(ctx, "takes_rotated", False)
                   and layer_ops.norm_linear_pays(rows, w) and layer_ops._rope_fits(cos, sin, x, c.head_dim))
        if rotated:
            src, norm = (x, n1.weight) if normed is None else (normed, None)
            qkv = layer_ops._qkv_linear(src, norm, n1.eps, w, a.qkv_proj.bias, cos, sin, c.num_heads + c.num_kv_heads)
        elif normed is not None:
            qkv = F.linear(normed, w, a.qkv_proj.bias)
        elif layer_ops.norm_linear_pays(rows, w):
            qkv = layer_ops._norm_linear(x, n1.weight, n1.eps, w, a.qkv_proj.bias)
        else:
            qkv = F.linear(layer_ops._rms_norm(x, n1.weight, n1.eps), w, a.qkv_proj.bias)
        out, w = a.attend(qkv, cos, sin, ctx, rotated), a.o_proj.weight
        if out.shape != (*x.shape[:2], c.q_size) or not layer_ops._operands(x, out):  # outputs of the context's own kind
            x = x + F.linear(out, w)
            return x + m(n2(x)), None
        w2 = m.gate_up_proj.weight
        if layer_ops.linear_residual_pays(rows, w):
            x = layer_ops._linear_residual(out, w, x)
            normed = None if layer_ops.norm_gate_up_pays(rows, w2) else layer_ops._rms_norm(x, n2.weight, n2.eps)
        else:
            x, normed = layer_ops._add_rms_norm(x, F.linear(out, w), n2.weight, n2.eps)
        if normed is None:
            act = layer_ops._norm_linear(x, n2.weight, n2.eps, w2, gate_up=True)
        else:
            act = m.gated(F.linear(normed, w2))
        w = m.down_proj.weight
        if (layer_ops.linear_residual_pays(rows, w) and act.shape == (*x.shape[:2], w.shape[1])
                and layer_ops._operands(x, act)):
            return layer_ops._linear_residual(act, w, x), None
        return x, F.linear(act, w)


_FORWARD = {cls: cls.forward for cls in (nn.Linear, RMSNorm, Attention, MLP, DecoderLayer)}


class Qwen2ForCausalLM(nn.Module):
    """Embedding -> decoder layers -> final norm; ``compute_logits`` applies the LM head."""

    def __init__(self, cfg: Qwen2Config) -> None:
        super().__init__()
        self.cfg = cfg
        self.embed_tokens = nn.Embedding(cfg.vocab_size, cfg.hidden_size)
        self.layers = nn.ModuleList(DecoderLayer(cfg, i) for i in range(cfg.num_layers))
        self.norm = RMSNorm(cfg.hidden_size, cfg.rms_norm_eps)
        self.lm_head = None if cfg.tie_word_embeddings else nn.Linear(cfg.hidden_size, cfg.vocab_size, bias=False)

    def forward(self, input_ids: torch.Tensor, positions: torch.Tensor, ctx: AttentionContext) -> torch.Tensor:
        x = self.embed_tokens(input_ids)
        cos, sin = rope_cos_sin(positions, self.cfg.head_dim, self.cfg.rope_theta, x.dtype)
        delta = None  # the last fused layer's residual add, left for the norm that follows it
        for layer in self.layers:
            if _plain(layer, DecoderLayer) and layer._fusable(x):
                x, delta = layer._fused(x, delta, cos, sin, ctx)
            else:
                x, delta = layer(x if delta is None else x + delta, cos, sin, ctx), None
        if delta is None:
            return self.norm(x)
        if _plain(self.norm, RMSNorm) and layer_ops.norm_usable(self.norm.weight, x, delta):
            return layer_ops._add_rms_norm(x, delta, self.norm.weight, self.norm.eps)[1]
        return self.norm(x + delta)

    def compute_logits(self, hidden: torch.Tensor) -> torch.Tensor:
        w = self.embed_tokens.weight if self.lm_head is None else self.lm_head.weight
        return F.linear(hidden, w)


def random_init_(model: Qwen2ForCausalLM, seed: int = 0, std: float = 0.02) -> Qwen2ForCausalLM:
    """Fill every weight in place from a seeded normal on its own device (norm weights stay 1)."""
    dev = next(model.parameters()).device
    gen = torch.Generator(device=dev).manual_seed(seed)
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name.endswith("norm.weight"):
                p.fill_(1.0)
            else:
                p.normal_(0.0, std, generator=gen)
    return model


def head_scale(head_dim: int) -> float:
    return 1.0 / math.sqrt(head_dim)
