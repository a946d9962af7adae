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
from torch.fx._symbolic_trace import is_fx_symbolic_tracing
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
            or torch._C._get_tracing_state() is not None or is_fx_symbolic_tracing() or torch.is_autocast_enabled("cuda"))


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


def _norm_fits(weight: torch.Tensor, x: torch.Tensor) -> bool:
    return weight.dim() == 1 and x.dim() >= 1 and weight.shape[0] == x.shape[-1] and _row_ok(x, _MAX_ROW_BYTES)


def norm_usable(weight: torch.Tensor, x: torch.Tensor, delta: torch.Tensor | None = None) -> bool:
    """Whether :func:`add_rms_norm` / :func:`rms_norm` take these (``delta`` of x's own shape)."""
    if not _open(x) or not _norm_fits(weight, x):
        return False
    if delta is None:
        return _operands(x, weight)
    return delta.shape == x.shape and _operands(x, delta, weight)


def _check(what: str, fits: bool, x: torch.Tensor, *others: torch.Tensor) -> None:
    """Raise unless the shapes fit (decided by the caller) and the tensors are dense, of one supported dtype and on
    one ROCm device: a kernel is given pointers and counts its rows itself. (Alignment is the C entry's to check.)

    Each function below has an underscored form without this check, for callers that have compared every shape and
    asked ``usable`` (2 to 3 us a call, four calls a layer)."""
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
    return _rms_norm(x, weight, eps)


def _rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
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
    return _add_rms_norm(x, delta, weight, eps)


def _add_rms_norm(x: torch.Tensor, delta: torch.Tensor, weight: torch.Tensor,
                  eps: float) -> tuple[torch.Tensor, torch.Tensor]:
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
    return _silu_mul(gate_up)


def _silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    inter = gate_up.shape[-1] // 2
    out = torch.empty((*gate_up.shape[:-1], inter), dtype=gate_up.dtype, device=gate_up.device)
    st = _native.load().mip_silu_mul(out.data_ptr(), gate_up.data_ptr(), gate_up.numel() // (2 * inter), inter,
                                     _DTYPE_CODES[gate_up.dtype], _stream_ptr(gate_up.device))
    if st:
        _native.check(st, "mip_silu_mul")
    return out


# Where the fused linear kernels beat the library's product and the separate kernels around it: a
# workgroup reads its rows of the input again for every 16 to 64 weight rows and K is split over its
# wavefronts alone, so they win while the rows are few, the weight small and K short. Lines between
# measured shapes (n x k by rows: fp16 | bf16, weights cold, graph replay, us, fused / library with the
# same elementwise work; linear + residual with the RMS norm that follows on both sides):
#   norm + linear     1152 x 896: 8 rows 4.2/7.7 | 4.5/8.7, 64 5.1/10.5 | 5.4/11.2, 256 9.9/10.4 | 10.2/11.3;
#                     4096 x 2048: 16 9.4/14.6 | 9.6/16.7; 2048 x 4096: 16 14.5/14.6 | 14.8/18.9;
#                     4608 x 3584: 8 - | 20.0/16.4; 2048 x 2048: 64 12.8/15.0 | 13.1/16.8;
#                     1024 x 4096: 32 14.2/14.7 | 14.6/15.5, 33 19.3/14.2 | 20.0/17.9;
#                     2048 x 1536: 96 12.6/12.4 | 12.9/13.8; 3072 x 1344: 65 18.9/16.6 | 19.5/18.0;
#                     1536 x 1024: 256 10.1/11.2 | 10.3/12.0; 1024 x 1536: 129 13.7/10.3 | 14.1/11.8
#   norm + gate + up  9728 x 896: 8 8.9/13.4 | 9.5/14.8, 64 16.1/17.0 | 16.6/18.5, 65 - | 27.0/18.4;
#                     22016 x 2048: 16 36.7/50.1 | 37.6/52.3; 16384 x 3072: 1 33.2/28.3 | 34.6/29.4;
#                     12288 x 1024: 17 20.4/17.8 | 20.2/19.2, 64 17.4/18.6 | 17.9/19.8;
#                     8192 x 1536: 33 20.1/16.8 | 20.5/18.4
#   linear + residual 896 x 896: 8 6.3/8.1 | 7.2/9.5, 256 9.2/10.5 | 10.0/11.8;
#                     896 x 4864: 8 13.2/15.8 | 14.0/21.1, 64 15.0/15.6 | 15.8/21.4;
#                     2048 x 2048: 64 15.5/15.9 | 17.4/18.6; 2048 x 2560: 33 16.4/13.5 | 18.5/16.3;
#                     1536 x 1536: 32 9.4/11.1 | 11.1/13.2, 33 (384 workgroups) 12.8/10.6 | 14.4/13.3;
#                     768 x 1344: 256 10.9/12.4 | 11.8/13.8; 512 x 2048: 256 12.2/10.7 | 12.9/11.5;
#                     3584 x 18944: 1 31.0/52.3 | 32.0/53.5, 16 46.0/52.5 | 47.2/54.0;
#                     5120 x 14336: 16 63.4/42.8 | 64.6/45.1
# At up to 16 rows the library's time of linear + residual jumps with k: over n <= 4096 the fused kernel
# is ahead for k up to 4864 and at 11008 and 18944, level at one row and behind at 8 to 16 rows for k =
# 8192 (3584 x 8192, 16 rows: 21.4/19.3 | 22.2/20.7) and 14336 (36.5/30.7 | 37.5/31.5).
_HALF = (torch.float16, torch.bfloat16)


def _linear_fits(rows: int, weight: torch.Tensor) -> bool:
    n, k = weight.shape
    return rows <= 256 and weight.dtype in _HALF and n % 16 == 0 and k % 32 == 0


def norm_linear_pays(rows: int, weight: torch.Tensor) -> bool:
    """Also the rule of :func:`qkv_linear`, which besides saves the rotary kernel (3 to 5 us)."""
    elements, k = ((8 << 20, 4096) if rows <= 16 else (4 << 20, 4096) if rows <= 32 else (4 << 20, 2048) if rows <= 64
                   else (3 << 20, 2048) if rows <= 96 else (3 << 19, 1024))
    return _linear_fits(rows, weight) and weight.numel() <= elements and weight.shape[1] <= k


def norm_gate_up_pays(rows: int, weight: torch.Tensor) -> bool:
    elements, k = ((48 << 20, 2048) if rows <= 16 else (9 << 20, 1024) if rows <= 32 else (12 << 20, 1152) if rows <= 64
                   else (0, 0))
    return _linear_fits(rows, weight) and weight.numel() <= elements and weight.shape[1] <= k


def linear_residual_pays(rows: int, weight: torch.Tensor) -> bool:
    if not _linear_fits(rows, weight):
        return False
    n, k = weight.shape
    if rows <= 16:
        return n <= 4096 and k <= 20480  # one round of 16-column workgroups on 256 CUs
    if rows <= 64:  # one round too; from n = 2048 on the tiles are 32 x 32
        return n * k < 9 << 19 and (n >= 2048 or (rows + 15) // 16 * (n // 16) <= 256)
    return n * k <= 1 << 20 and k <= 1536


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
    return _norm_linear(x, norm, eps, weight, bias, gate_up)


def _norm_linear(x: torch.Tensor, norm: torch.Tensor, eps: float, weight: torch.Tensor,
                 bias: torch.Tensor | None = None, gate_up: bool = False) -> torch.Tensor:
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
    return _open(x) and _rope_fits(cos, sin, x, head_dim)


def _rope_fits(cos: torch.Tensor, sin: torch.Tensor, x: torch.Tensor, head_dim: int) -> bool:
    return (cos.shape == sin.shape == (x.shape[0], 1, x.shape[1], head_dim) and head_dim % 16 == 0
            and _operands(x, cos, sin))


def qkv_linear(x: torch.Tensor, norm: torch.Tensor | None, eps: float, weight: torch.Tensor, bias: torch.Tensor | None,
               cos: torch.Tensor, sin: torch.Tensor, rot_heads: int) -> torch.Tensor:
    """:func:`norm_linear` (of x itself where ``norm`` is None) with the rotary embedding applied to the first
    ``rot_heads`` heads of its output; cos, sin ``[B, 1, T, head_dim]``. The rotation is
    :func:`engine.paged_ops.rope_kv_append`'s, bit for bit."""
    extra = tuple(t for t in (norm, bias) if t is not None)
    _check("qkv_linear", _weight(weight, x) and x.dim() == 3 and (norm is None or norm.shape == (x.shape[-1],))
           and (bias is None or bias.shape == weight.shape[:1]) and cos.dim() == 4
           and cos.shape == sin.shape == (x.shape[0], 1, x.shape[1], cos.shape[-1]), x, weight, cos, sin, *extra)
    return _qkv_linear(x, norm, eps, weight, bias, cos, sin, rot_heads)


def _qkv_linear(x: torch.Tensor, norm: torch.Tensor | None, eps: float, weight: torch.Tensor, bias: torch.Tensor | None,
                cos: torch.Tensor, sin: torch.Tensor, rot_heads: int) -> torch.Tensor:
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
    return _linear_residual(a, weight, residual)


def _linear_residual(a: torch.Tensor, weight: torch.Tensor, residual: torch.Tensor) -> torch.Tensor:
    n, k = weight.shape
    out = torch.empty_like(residual)
    st = _native.load().mip_linear_residual(out.data_ptr(), a.data_ptr(), weight.data_ptr(), residual.data_ptr(),
                                            a.numel() // k, n, k, _DTYPE_CODES[a.dtype], _stream_ptr(a.device))
    if st:
        _native.check(st, "mip_linear_residual")
    return out
