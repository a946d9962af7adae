"""Fused kernels of a decoder layer, used by :mod:`engine.model` where they apply.

``usable`` is the rule: plain contiguous tensors of one supported dtype on the current ROCm
device, with nothing recording, transforming or tracing the call. Everything else (CPU tensors,
autograd, torch.func, autocast, tensor subclasses, odd layouts) keeps the torch ops, which
compute the same values. Each function checks its operands on the host and raises for those
that its kernel cannot read.
"""

from __future__ import annotations

import torch
import torch.overrides
from torch.fx._symbolic_trace import is_fx_tracing as _is_fx_tracing
from torch.utils._device import DeviceContext

from . import _native
from .paged_ops import _DTYPE_CODES, _require_device, _stream_ptr, dtype_code

_FWD_AD = torch.autograd.forward_ad
_PLAIN = (torch.Tensor, torch.nn.Parameter)
_MAX_ROW_BYTES = 32768


def _function_mode() -> bool:
    """Whether a mode sees torch calls. A default device (``torch.set_default_device``, ``with torch.device(..)``) is a
    mode too, but one that only fills in the device of calls that name none."""
    return torch._C._len_torch_function_stack() > 0 and any(
        type(m) is not DeviceContext for m in torch.overrides._get_current_function_mode_stack())


def _observed() -> bool:
    """Whether something other than the plain eager dispatch would see a torch op called now."""
    return (torch.compiler.is_compiling()  # first: a compiler that traces this function stops reading here
            or _function_mode() or torch._C._len_torch_dispatch_stack() > 0
            or torch._C._functorch.peek_interpreter_stack() is not None or _FWD_AD._current_level >= 0
            or torch._C._get_tracing_state() is not None or _is_fx_tracing() or torch.is_autocast_enabled("cuda"))


def _open(x: torch.Tensor) -> bool:
    """Whether this device tensor's op may be taken over at all (asked before anything about its sizes: a symbolic
    tracer's stand-in for a tensor answers no such question)."""
    return type(x) in _PLAIN and x.is_cuda and x.dtype in _DTYPE_CODES and not _observed()


def _operands(x: torch.Tensor, *others: torch.Tensor) -> bool:
    """Whether the kernels can read these: dense, 16-byte aligned, one dtype, on the current device, no gradient."""
    grad = torch.is_grad_enabled()
    for t in (x, *others):
        if (type(t) not in _PLAIN or t.dtype != x.dtype or t.device != x.device or not t.is_contiguous()
                or t.data_ptr() % 16 or (grad and t.requires_grad) or t.is_neg()):
            return False
    return x.device.index == torch.cuda.current_device()


def usable(x: torch.Tensor, *others: torch.Tensor) -> bool:
    """Whether the fused kernels may take these operands."""
    return _open(x) and _operands(x, *others)


def _row_ok(t: torch.Tensor, limit: int) -> bool:
    if t.dim() < 1 or t.numel() == 0:
        return False
    nbytes = t.shape[-1] * t.element_size()
    return nbytes % 16 == 0 and nbytes <= limit and t.numel() // t.shape[-1] < 1 << 31


def norm_usable(weight: torch.Tensor, x: torch.Tensor, delta: torch.Tensor | None = None) -> bool:
    """Whether :func:`add_rms_norm` / :func:`rms_norm` take these (``delta`` of x's own shape)."""
    if not _open(x):
        return False
    if weight.dim() != 1 or x.dim() < 1 or weight.shape[0] != x.shape[-1] or not _row_ok(x, _MAX_ROW_BYTES):
        return False
    if delta is None:
        return _operands(x, weight)
    return delta.shape == x.shape and _operands(x, delta, weight)


def _check(what: str, fits: bool, x: torch.Tensor, *others: torch.Tensor) -> None:
    """Raise unless the shapes fit (decided by the caller) and the tensors are dense, of one supported dtype and on
    one ROCm device: a kernel is given pointers and counts its rows itself. (Alignment is the C entry's to check.)"""
    if not fits or x.numel() >= x.shape[-1] << 31:
        raise ValueError(f"{what}: shapes do not fit: {', '.join(str(tuple(t.shape)) for t in (x, *others))}")
    dtype_code(x.dtype)
    for t in (x, *others):
        if t.dtype != x.dtype:
            raise TypeError(f"{what}: operands must share one dtype")
        if not t.is_contiguous() or t.device != x.device:
            raise ValueError(f"{what}: operands must be contiguous and on one device")
    _require_device(x)


def _rows_of(x: torch.Tensor, width: int) -> bool:
    return x.dim() >= 1 and x.shape[-1] == width > 0


def _weight(w: torch.Tensor, x: torch.Tensor) -> bool:
    return w.dim() == 2 and w.shape[0] > 0 and _rows_of(x, w.shape[1])


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    """``weight * (x.float() * rsqrt(mean(x.float()^2) + eps)).to(dtype)`` in one launch."""
    _check("rms_norm", weight.dim() == 1 and _rows_of(x, weight.shape[0]), x, weight)
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
    _check("add_rms_norm", weight.dim() == 1 and _rows_of(x, weight.shape[0]) and delta.shape == x.shape,
           x, delta, weight)
    s, out = torch.empty_like(x), torch.empty_like(x)
    st = _native.load().mip_add_rms_norm(out.data_ptr(), s.data_ptr(), x.data_ptr(), delta.data_ptr(),
                                         weight.data_ptr(), x.numel() // x.shape[-1], x.shape[-1], eps,
                                         _DTYPE_CODES[x.dtype], _stream_ptr(x.device))
    if st:
        _native.check(st, "mip_add_rms_norm")
    return s, out


def rope_tables(positions: torch.Tensor, head_dim: int, theta: float,
                dtype: torch.dtype) -> tuple[torch.Tensor, torch.Tensor] | None:
    """cos/sin ``[B, 1, T, D]`` for ``positions [B, T]`` in one launch, or None where it does not apply."""
    if (type(positions) is not torch.Tensor or not positions.is_cuda or _observed() or positions.dtype != torch.int64
            or positions.dim() != 2 or not positions.is_contiguous() or dtype not in _DTYPE_CODES or head_dim % 2
            or type(theta) not in (float, int) or theta <= 0 or not 0 < positions.numel() * head_dim < 1 << 31
            or positions.device.index != torch.cuda.current_device()):
        return None
    b, t = positions.shape
    cos, sin = (torch.empty((b, 1, t, head_dim), dtype=dtype, device=positions.device) for _ in range(2))
    st = _native.load().mip_rope_tables(cos.data_ptr(), sin.data_ptr(), positions.data_ptr(), b * t, head_dim, theta,
                                        _DTYPE_CODES[dtype], _stream_ptr(positions.device))
    if st:
        _native.check(st, "mip_rope_tables")
    return cos, sin


def silu_mul_usable(gate_up: torch.Tensor) -> bool:
    if not _open(gate_up) or gate_up.dim() < 1 or gate_up.shape[-1] % 2 or gate_up.numel() == 0:
        return False
    half = gate_up.shape[-1] // 2 * gate_up.element_size()
    return half % 16 == 0 and gate_up.numel() * gate_up.element_size() // 32 < 1 << 31 and _operands(gate_up)


def silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    """``silu(gate) * up`` of the halves of the last dimension, in one launch."""
    _check("silu_mul", gate_up.dim() >= 1 and gate_up.shape[-1] > 0 and gate_up.shape[-1] % 2 == 0, gate_up)
    inter = gate_up.shape[-1] // 2
    out = torch.empty((*gate_up.shape[:-1], inter), dtype=gate_up.dtype, device=gate_up.device)
    st = _native.load().mip_silu_mul(out.data_ptr(), gate_up.data_ptr(), gate_up.numel() // (2 * inter), inter,
                                     _DTYPE_CODES[gate_up.dtype], _stream_ptr(gate_up.device))
    if st:
        _native.check(st, "mip_silu_mul")
    return out


# Where the fused linear kernels beat the library's product and the separate kernels around it: a
# workgroup reads its rows of the input again for every 16 to 64 weight rows, so they win while
# the rows are few or the weight small. Lines between measured shapes (bf16, weights cold, graph
# replay, us, fused against library), n x k by rows:
#   norm + linear     1152 x 896: 4.5/8.6 at 8 rows, 5.7/11.2 at 64, 10.1/11.2 at 256;
#                     2560 x 2048: 8.8/16.2 at 16, 13.2/16.6 at 65, 26.4/19.7 at 128;
#                     2048 x 1536: 12.7/13.8 at 128, 15.5/14.6 at 256; 4608 x 3584: 20.0/16.4 at 8
#   norm + gate + up  9728 x 896: 9.3/14.6 at 8, 16.3/18.3 at 64, 27.0/18.4 at 65;
#                     17920 x 1536: 28.7/47.4 at 16, 35.7/26.1 at 32; 22016 x 2048: 37.4/52.4 at 16;
#                     37888 x 3584: 104/65 at 8
#   linear + residual 896 x 896: 3.8/8.5 at 8, 6.2/9.7 at 256; 896 x 4864: 10.5/20.3 at 8,
#                     12.0/19.1 at 64, 17.8/15.5 at 96; 2048 x 2048: 11.7/13.8 at 64;
#                     3584 x 3584: 10.9/15.1 at 16, 18.7/14.9 at 32; 3584 x 18944: 39.0/48.7 at 16
_HALF = (torch.float16, torch.bfloat16)


def _linear_fits(rows: int, weight: torch.Tensor) -> bool:
    n, k = weight.shape
    return rows <= 256 and weight.dtype in _HALF and n % 16 == 0 and k % 32 == 0


def norm_linear_pays(rows: int, weight: torch.Tensor) -> bool:
    limit = 8 << 20 if rows <= 16 else 4 << 20 if rows <= 96 else 3 << 19
    return _linear_fits(rows, weight) and weight.numel() <= limit


def qkv_linear_pays(rows: int, weight: torch.Tensor, normed: bool) -> bool:
    """As :func:`norm_linear_pays`, with the rotary kernel that the library's product leaves to be run (3 to 5 us);
    ``normed``: x is normed already (1152 x 896 at 256 rows: 10.1 us with the rotation against 10.6 + 5.0, under
    the profiler; 2048 x 1536 at 256 rows 12.9 against 9.9 + 5.0, not worth a rule of its own)."""
    return norm_linear_pays(rows, weight) or (normed and _linear_fits(rows, weight) and weight.numel() <= 3 << 19)


def norm_gate_up_pays(rows: int, weight: torch.Tensor) -> bool:
    limit = 48 << 20 if rows <= 16 else 12 << 20 if rows <= 64 else 0
    return _linear_fits(rows, weight) and weight.numel() <= limit


def linear_residual_pays(rows: int, weight: torch.Tensor) -> bool:
    if not _linear_fits(rows, weight):
        return False
    return rows <= 16 or weight.numel() <= (5 << 20 if rows <= 64 else 1 << 20)


def norm_linear(x: torch.Tensor, norm: torch.Tensor, eps: float, weight: torch.Tensor, bias: torch.Tensor | None = None,
                gate_up: bool = False) -> torch.Tensor:
    """The RMS norm of x's rows through a linear layer, in one launch.

    With ``gate_up`` the weight holds gate rows, then as many up rows, and the result is
    ``silu(gate) * up``.
    """
    extra = () if bias is None else (bias,)
    _check("norm_linear", _weight(weight, x) and norm.shape == (x.shape[-1],)
           and (bias is None or bias.shape == weight.shape[:1])
           and not (gate_up and (extra or weight.shape[0] % 2)), x, weight, norm, *extra)
    n, k = weight.shape
    out = torch.empty((*x.shape[:-1], n // 2 if gate_up else n), dtype=x.dtype, device=x.device)
    st = _native.load().mip_norm_linear(out.data_ptr(), x.data_ptr(), norm.data_ptr(), eps, weight.data_ptr(),
                                        None if bias is None else bias.data_ptr(), x.numel() // k, n, k, int(gate_up),
                                        _DTYPE_CODES[x.dtype], _stream_ptr(x.device))
    if st:
        _native.check(st, "mip_norm_linear")
    return out


def rope_usable(cos: torch.Tensor, sin: torch.Tensor, x: torch.Tensor, head_dim: int) -> bool:
    """Whether :func:`qkv_linear` can take these rotary tables for rows ``x [B, T, hidden]``."""
    return (cos.shape == sin.shape == (x.shape[0], 1, x.shape[1], head_dim) and head_dim % 16 == 0
            and usable(x, cos, sin))


def qkv_linear(x: torch.Tensor, norm: torch.Tensor | None, eps: float, weight: torch.Tensor, bias: torch.Tensor | None,
               cos: torch.Tensor, sin: torch.Tensor, rot_heads: int) -> torch.Tensor:
    """:func:`norm_linear` (of x itself where ``norm`` is None) with the rotary embedding applied to the first
    ``rot_heads`` heads of its output; cos, sin ``[B, 1, T, head_dim]``. The rotation is
    :func:`engine.paged_ops.rope_kv_append`'s, bit for bit."""
    extra = tuple(t for t in (norm, bias) if t is not None)
    _check("qkv_linear", _weight(weight, x) and x.dim() == 3 and (norm is None or norm.shape == (x.shape[-1],))
           and (bias is None or bias.shape == weight.shape[:1]) and cos.dim() == 4
           and cos.shape == sin.shape == (x.shape[0], 1, x.shape[1], cos.shape[-1]), x, weight, cos, sin, *extra)
    n, k = weight.shape
    d = cos.shape[-1]
    out = torch.empty((*x.shape[:-1], n), dtype=x.dtype, device=x.device)
    st = _native.load().mip_qkv_linear(out.data_ptr(), x.data_ptr(), None if norm is None else norm.data_ptr(), eps,
                                       weight.data_ptr(), None if bias is None else bias.data_ptr(), cos.data_ptr(),
                                       sin.data_ptr(), d, x.numel() // k, n, k, d, rot_heads, _DTYPE_CODES[x.dtype],
                                       _stream_ptr(x.device))
    if st:
        _native.check(st, "mip_qkv_linear")
    return out


def linear_residual(a: torch.Tensor, weight: torch.Tensor, residual: torch.Tensor) -> torch.Tensor:
    """``residual + a @ weight.T`` in one launch."""
    _check("linear_residual", _weight(weight, a) and residual.shape == (*a.shape[:-1], weight.shape[0]),
           a, weight, residual)
    n, k = weight.shape
    out = torch.empty_like(residual)
    st = _native.load().mip_linear_residual(out.data_ptr(), a.data_ptr(), weight.data_ptr(), residual.data_ptr(),
                                            a.numel() // k, n, k, _DTYPE_CODES[a.dtype], _stream_ptr(a.device))
    if st:
        _native.check(st, "mip_linear_residual")
    return out
