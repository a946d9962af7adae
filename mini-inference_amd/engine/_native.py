"""ctypes binding of libmipaged.so, the C-ABI HIP library (declared in include/mipaged.h).

Loading is lazy and strict: any use of a kernel without the built library, or with
tensors that are not on a ROCm device, raises. There is no CPU fallback.
"""

from __future__ import annotations

import ctypes
import os
from pathlib import Path

LIB_PATH = Path(__file__).resolve().parent / "libmipaged.so"

MIP_F32, MIP_F16, MIP_BF16 = 0, 1, 2
MIP_OK, MIP_E2BIG, MIP_EINVAL, MIP_EUNSUPPORTED = 0, -7, -22, -95
MIP_NOALLOC_SCRATCH_BYTES = 32 << 20
MIP_ALGO = {"auto": 0, "valu": 1, "mfma": 2, "stream": 3}

EXPORTED = (
    "mip_version",
    "mip_status_string",
    "mip_set_decode_algo",
    "mip_kv_append",
    "mip_rope_kv_append",
    "mip_paged_decode",
    "mip_paged_decode_append",
    "mip_paged_decode_append_noalloc",
    "mip_paged_decode_workspace",
    "mip_paged_decode_plan",
    "mip_paged_decode_plan_bytes",
    "mip_paged_prefill",
    "mip_copy_blocks",
    "mip_copy_blocks_host",
    "mip_prefill_index",
    "mip_decode_prepare",
    "mip_rope_tables",
    "mip_decode_step_append",
    "mip_decode_step_attend",
    "mip_rope_step_append",
    "mip_prefill_step_append",
    "mip_prefill_step_attend",
    "mip_add_rms_norm",
    "mip_silu_mul",
    "mip_norm_linear",
    "mip_qkv_linear",
    "mip_linear_residual",
)

# Measurement helpers in the same library (include/mipaged_probe.h), outside the drop-in ABI.
PROBE_EXPORTED = ("mip_hbm_read_probe",)

_c = ctypes
_i32, _i64, _sz, _vp, _f32 = _c.c_int32, _c.c_int64, _c.c_size_t, _c.c_void_p, _c.c_float


class DecodeStep(_c.Structure):
    """``mip_decode_step``: what every layer's decode call of one step shares."""

    _fields_ = [(n, _i64) for n in ("k_stride_tok", "k_stride_head", "v_stride_tok", "v_stride_head")] + [
        ("slot_mapping", _vp)] + [(n, _i64) for n in ("out_stride_b", "out_stride_h", "q_stride_b", "q_stride_h",
                                                      "num_cache_blocks")] + [
        ("block_tables", _vp), ("bt_stride", _i64), ("context_lens", _vp), ("workspace", _vp), ("workspace_bytes", _sz),
        ("plan", _vp), ("plan_bytes", _sz)] + [
        (n, _i32) for n in ("batch", "num_heads", "num_kv_heads", "head_dim", "block_size", "max_blocks_per_seq",
                            "dtype")] + [("scale", _f32)]


class RopeStep(_c.Structure):
    """``mip_rope_step``: what every layer's rotary embedding + append call of one step shares."""

    _fields_ = [(n, _i64) for n in ("q_stride_tok", "q_stride_head", "k_stride_tok", "k_stride_head", "v_stride_tok",
                                    "v_stride_head", "cs_stride_tok", "num_cache_blocks")] + [("slot_mapping", _vp)] + [
        (n, _i32) for n in ("n_tokens", "num_heads", "num_kv_heads", "head_dim", "block_size", "dtype")]


class PrefillStep(_c.Structure):
    """``mip_prefill_step``: what every layer's packed prefill calls of one step share."""

    _fields_ = [(n, _i64) for n in ("k_stride_tok", "k_stride_head", "v_stride_tok", "v_stride_head")] + [
        ("slot_mapping", _vp)] + [(n, _i64) for n in ("out_stride_tok", "out_stride_head", "q_stride_tok",
                                                      "q_stride_head", "num_cache_blocks")] + [
        ("block_tables", _vp), ("bt_stride", _i64), ("cu_q", _vp), ("ctx_start", _vp)] + [
        (n, _i32) for n in ("n_tokens", "num_seqs", "max_q_len", "num_heads", "num_kv_heads", "head_dim", "block_size",
                            "max_blocks_per_seq", "dtype")] + [("scale", _f32)]


_SIGNATURES = {
    "mip_version": (_c.c_int, []),
    "mip_status_string": (_c.c_char_p, [_c.c_int]),
    "mip_set_decode_algo": (_c.c_int, [_i32]),
    "mip_kv_append": (
        _c.c_int,
        [_vp, _vp, _i64, _i64, _i64, _i64, _vp, _vp, _i64, _vp, _i32, _i32, _i32, _i32, _i32, _vp],
    ),
    "mip_rope_kv_append": (
        _c.c_int,
        [_vp, _i64, _i64, _vp, _i64, _i64, _vp, _i64, _i64, _vp, _vp, _i64,
         _vp, _vp, _i64, _vp, _i32, _i32, _i32, _i32, _i32, _i32, _vp],
    ),
    "mip_paged_decode": (
        _c.c_int,
        [_vp, _i64, _i64, _vp, _i64, _i64, _vp, _vp, _i64, _vp, _i64, _vp,
         _i32, _i32, _i32, _i32, _i32, _i32, _f32, _vp, _sz, _vp, _sz, _i32, _vp],
    ),
    "mip_paged_decode_append": (
        _c.c_int,
        [_vp, _vp, _i64, _i64, _i64, _i64, _vp,
         _vp, _i64, _i64, _vp, _i64, _i64, _vp, _vp, _i64, _vp, _i64, _vp,
         _i32, _i32, _i32, _i32, _i32, _i32, _f32, _vp, _sz, _vp, _sz, _i32, _vp],
    ),
    "mip_paged_decode_append_noalloc": (
        _c.c_int,
        [_vp, _vp, _i64, _i64, _i64, _i64, _vp,
         _vp, _i64, _i64, _vp, _i64, _i64, _vp, _vp, _i64, _vp, _i64, _vp,
         _i32, _i32, _i32, _i32, _i32, _i32, _f32, _vp, _sz, _i32, _vp],
    ),
    "mip_paged_decode_workspace": (_sz, [_i32, _i32, _i32, _i32, _i32, _i32, _i32]),
    "mip_paged_decode_plan_bytes": (_sz, [_i32, _i32, _i32, _i32, _i32, _i32, _i32]),
    "mip_paged_decode_plan": (
        _c.c_int,
        [_vp, _vp, _i64, _i32, _i32, _i32, _i32, _i32, _i32, _i32, _vp, _sz, _vp],
    ),
    "mip_paged_prefill": (
        _c.c_int,
        [_vp, _i64, _i64, _vp, _i64, _i64, _vp, _vp, _i64, _vp, _i64, _vp, _vp,
         _i32, _i32, _i32, _i32, _i32, _i32, _i32, _f32, _i32, _vp],
    ),
    "mip_decode_step_append": (_c.c_int, [_vp] * 8),
    "mip_decode_step_attend": (_c.c_int, [_vp] * 6),
    "mip_rope_step_append": (_c.c_int, [_vp] * 9),
    "mip_prefill_step_append": (_c.c_int, [_vp] * 6),
    "mip_prefill_step_attend": (_c.c_int, [_vp] * 6),
    "mip_decode_prepare": (_c.c_int, [_vp, _i64, _vp, _vp, _i32, _vp, _vp, _vp, _i64, _i32, _vp, _vp, _i32, _i32, _vp]),
    "mip_rope_tables": (_c.c_int, [_vp, _vp, _vp, _i32, _i32, _f32, _i32, _vp]),
    "mip_prefill_index": (_c.c_int, [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i32, _i32, _i32, _vp]),
    "mip_copy_blocks": (_c.c_int, [_vp, _vp, _vp, _i32, _i32, _i64, _i64, _vp]),
    "mip_copy_blocks_host": (_c.c_int, [_vp, _vp, _vp, _i32, _i32, _i64, _i64, _vp]),
    "mip_add_rms_norm": (_c.c_int, [_vp, _vp, _vp, _vp, _vp, _i32, _i32, _f32, _i32, _vp]),
    "mip_silu_mul": (_c.c_int, [_vp, _vp, _i32, _i32, _i32, _vp]),
    "mip_norm_linear": (_c.c_int, [_vp, _vp, _vp, _f32, _vp, _vp, _i32, _i32, _i32, _i32, _i32, _vp]),
    "mip_qkv_linear": (_c.c_int, [_vp, _vp, _vp, _f32, _vp, _vp, _vp, _vp, _i64, _i32, _i32, _i32, _i32, _i32, _i32, _vp]),
    "mip_linear_residual": (_c.c_int, [_vp, _vp, _vp, _vp, _i32, _i32, _i32, _i32, _vp]),
    "mip_hbm_read_probe": (_c.c_int, [_vp, _i64, _vp, _i64, _i32, _vp, _i32, _i32, _vp]),
}

_lib: ctypes.CDLL | None = None


class NativeLibraryMissing(RuntimeError):
    pass


class NativeError(RuntimeError):
    pass


def load(path: str | os.PathLike | None = None) -> ctypes.CDLL:
    """Load (once) and return the library, with argument types set for every entry point."""
    global _lib
    if _lib is not None and path is None:
        return _lib
    p = Path(path) if path is not None else LIB_PATH
    if not p.exists():
        raise NativeLibraryMissing(
            f"{p} is not built; run `python mini-inference_amd/build.py` (or __graft_entry__.build())"
        )
    lib = ctypes.CDLL(str(p))
    for name, (res, args) in _SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = res
        fn.argtypes = args
    if path is None:
        _lib = lib
    return lib


def set_decode_algo(name: str) -> str:
    """Force the decode attention algorithm ("auto", "valu", "mfma", "stream"); returns the previous one.

    Process-wide (``mip_set_decode_algo``); meant for kernel comparisons and tests.
    """
    prev = load().mip_set_decode_algo(MIP_ALGO[name])
    if prev < 0:
        raise NativeError(f"mip_set_decode_algo({name!r}) failed: status {prev}")
    return next(k for k, v in MIP_ALGO.items() if v == prev)


def check(status: int, what: str) -> None:
    if status != MIP_OK:
        msg = load().mip_status_string(status).decode()
        raise NativeError(f"{what} failed: status {status} ({msg})")
