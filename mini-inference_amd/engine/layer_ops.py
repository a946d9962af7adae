"""Fused elementwise kernels of a decoder layer, used by :mod:`engine.model` where they apply.

``usable`` is the rule: plain contiguous tensors of one supported dtype on the current ROCm
device, with nothing recording, transforming or tracing the call. Everything else (CPU tensors,
autograd, torch.func, autocast, tensor subclasses, odd layouts) keeps the torch ops, which
compute the same values.
"""

from __future__ import annotations

import torch

from . import _native
from .paged_ops import _DTYPE_CODES, _stream_ptr

_FWD_AD = torch.autograd.forward_ad
_PLAIN = (torch.Tensor, torch.nn.Parameter)
_MAX_ROW_BYTES = 32768


def _observed() -> bool:
    """Whether something other than the plain eager dispatch would see a torch op called now."""
    return (torch._C._len_torch_function_stack() > 0 or torch._C._len_torch_dispatch_stack() > 0
            or torch._C._functorch.peek_interpreter_stack() is not None or _FWD_AD._current_level >= 0
            or torch._C._get_tracing_state() is not None or torch.compiler.is_compiling()
            or torch.is_autocast_enabled("cuda"))


def usable(*tensors: torch.Tensor) -> bool:
    """Whether the fused kernels may take these operands (16-byte aligned, dense, one dtype and device)."""
    x = tensors[0]
    if not x.is_cuda or x.dtype not in _DTYPE_CODES or _observed():
        return False
    grad = torch.is_grad_enabled()
    for t in tensors:
        if (type(t) not in _PLAIN or t.dtype != x.dtype or t.device != x.device or not t.is_contiguous()
                or t.data_ptr() % 16 or (grad and t.requires_grad) or t.is_neg()):
            return False
    return x.device.index == torch.cuda.current_device()


def _row_ok(t: torch.Tensor, limit: int | None = None) -> bool:
    if t.dim() < 1 or t.numel() == 0:
        return False
    nbytes = t.shape[-1] * t.element_size()
    return nbytes % 16 == 0 and (limit is None or nbytes <= limit) and t.numel() // t.shape[-1] < 1 << 31


def norm_usable(weight: torch.Tensor, x: torch.Tensor, delta: torch.Tensor | None = None) -> bool:
    """Whether :func:`add_rms_norm` / :func:`rms_norm` take these (``delta`` of x's own shape)."""
    if weight.dim() != 1 or x.dim() < 1 or weight.shape[0] != x.shape[-1] or not _row_ok(x, _MAX_ROW_BYTES):
        return False
    if delta is None:
        return usable(x, weight)
    return delta.shape == x.shape and usable(x, delta, weight)


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    """``weight * (x.float() * rsqrt(mean(x.float()^2) + eps)).to(dtype)`` in one launch."""
    out = torch.empty_like(x)
    st = _native.load().mip_add_rms_norm(out.data_ptr(), None, x.data_ptr(), None, weight.data_ptr(),
                                         x.numel() // x.shape[-1], x.shape[-1], eps, _DTYPE_CODES[x.dtype],
                                         _stream_ptr(x.device))
    if st:
        _native.check(st, "mip_add_rms_norm")
    return out


def add_rms_norm(x: torch.Tensor, delta: torch.Tensor, weight: torch.Tensor,
                 eps: float) -> tuple[torch.Tensor, torch.Tensor]:
    """``s = x + delta`` and the RMS norm of ``s``, in one launch; returns ``(s, normed)``."""
    s, out = torch.empty_like(x), torch.empty_like(x)
    st = _native.load().mip_add_rms_norm(out.data_ptr(), s.data_ptr(), x.data_ptr(), delta.data_ptr(),
                                         weight.data_ptr(), x.numel() // x.shape[-1], x.shape[-1], eps,
                                         _DTYPE_CODES[x.dtype], _stream_ptr(x.device))
    if st:
        _native.check(st, "mip_add_rms_norm")
    return s, out


def silu_mul_usable(gate_up: torch.Tensor) -> bool:
    if gate_up.dim() < 1 or gate_up.shape[-1] % 2 or gate_up.numel() == 0:
        return False
    half = gate_up.shape[-1] // 2 * gate_up.element_size()
    return half % 16 == 0 and gate_up.numel() * gate_up.element_size() // 32 < 1 << 31 and usable(gate_up)


def silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    """``silu(gate) * up`` of the halves of the last dimension, in one launch."""
    inter = gate_up.shape[-1] // 2
    out = torch.empty((*gate_up.shape[:-1], inter), dtype=gate_up.dtype, device=gate_up.device)
    st = _native.load().mip_silu_mul(out.data_ptr(), gate_up.data_ptr(), gate_up.numel() // (2 * inter), inter,
                                     _DTYPE_CODES[gate_up.dtype], _stream_ptr(gate_up.device))
    if st:
        _native.check(st, "mip_silu_mul")
    return out
