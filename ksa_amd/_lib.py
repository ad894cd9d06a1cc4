"""ctypes binding of libksa_hip.so.  There is no fallback: if the library is missing
or does not load, every operator of this package raises."""
from __future__ import annotations

import contextlib
import ctypes
import functools
import os
import warnings

import torch  # noqa: F401  (must be imported first so that its HIP runtime is the one in the process)

_HERE = os.path.dirname(os.path.abspath(__file__))
# KSA_AMD_LIB selects another build of the same library (e.g. a profiling variant)
LIB_PATH = os.environ.get("KSA_AMD_LIB") or os.path.join(_HERE, "libksa_hip.so")
_lib = None
# the native front of the hottest calls (csrc/ksa_fast.cpp; `_GeneralWay` where it does not load); what it calls, in the order
# of its `bind`
fast = None
_FAST = ("ksa_block_index", "ksa_decode_splits", "ksa_decode_workspace_bytes", "ksa_decode_fwd", "ksa_prefill_chunks_fwd",
         "ksa_pre_attention", "ksa_decode_wide_splits", "ksa_decode_wide_fwd")

_i32p = ctypes.POINTER(ctypes.c_int32)
_i64p = ctypes.POINTER(ctypes.c_int64)
_vp = ctypes.c_void_p
_int = ctypes.c_int

_SIGNATURES = {
    "ksa_version": (_int, []),
    "ksa_error_string": (ctypes.c_char_p, [_int]),
    "ksa_device_cu_count": (_int, []),
    "ksa_block_index": (_int, [_int] * 9 + [_vp] * 4 + [_vp]),
    "ksa_prefill_fwd": (_int, [_vp] * 5 + [_int] * 6 + [_i64p] * 3 + [_int] * 6 + [_vp] * 4
                        + [_int, ctypes.c_float, _int, _vp, _vp]),
    "ksa_prefill_chunks_fwd": (_int, [_vp] * 5 + [_int] * 6 + [_i64p] * 3 + [_int] * 4
                               + [ctypes.c_float, _int, _vp, _vp]),
    "ksa_decode_workspace_bytes": (ctypes.c_size_t, [_int] * 6),
    "ksa_decode_auto_splits": (_int, [_int] * 3),
    "ksa_decode_splits": (_int, [_int] * 6),
    "ksa_decode_fwd": (_int, [_vp] * 6 + [_int] * 8 + [_i64p] * 4
                       + [ctypes.c_float, _int, _vp, ctypes.c_size_t, _vp]),
    "ksa_decode_qkv_fwd": (_int, [_vp, _int] + [_vp] * 4 + [ctypes.c_longlong, ctypes.c_float] + [_vp] * 4 + [_int]
                           + [_vp] * 2 + [_int] * 7 + [_i64p] * 3 + [ctypes.c_float, _int, _vp, ctypes.c_size_t, _vp]),
    "ksa_decode_wide_splits": (_int, [_int] * 6),
    "ksa_decode_wide_fwd": (_int, [_vp] * 6 + [_int] * 8 + [_i64p] * 4
                       + [ctypes.c_float, _int, _vp, ctypes.c_size_t, _vp]),
    "ksa_decode_qkv_wide_fwd": (_int, [_vp, _int] + [_vp] * 4 + [ctypes.c_longlong, ctypes.c_float] + [_vp] * 4 + [_int]
                           + [_vp] * 2 + [_int] * 7 + [_i64p] * 3 + [ctypes.c_float, _int, _vp, ctypes.c_size_t, _vp]),
    "ksa_decode_noalloc_max_workspace_bytes": (ctypes.c_size_t, []),
    "ksa_decode_fwd_noalloc": (_int, [_vp] * 6 + [_int] * 8 + [_i64p] * 4 + [ctypes.c_float, _int, _vp]),
    "ksa_decode_weights_workspace_bytes": (ctypes.c_size_t, [_int] * 4),
    "ksa_decode_weights": (_int, [_vp] * 6 + [_int] * 9 + [_i64p, _i64p, _vp] + [ctypes.c_float, _vp, ctypes.c_size_t, _vp]),
    "ksa_decode_boundary_workspace_bytes": (ctypes.c_size_t, [_int] * 6),
    "ksa_decode_boundary_fwd": (_int, [_vp] * 6 + [_int, _int, _vp, _vp] + [_int] * 8 + [_i64p] * 4
                                + [ctypes.c_float, _int, _vp, ctypes.c_size_t, _vp]),
    "ksa_copy_rows_multi": (_int, [_int, _vp, _vp, _vp, _vp, _vp, _vp, _int, _int, _int, _vp, _vp, _vp]),
    "ksa_copy_rows_runs": (_int, [_int] + [_vp] * 5 + [_int] + [_vp] * 2 + [_int] * 3 + [_vp] * 3),
    "ksa_expand_prompt": (_int, [_vp, ctypes.c_longlong] + [_int] * 4 + [ctypes.c_longlong, _int, _int, _vp, _int]
                          + [_vp] * 4 + [_int, _vp]),
    "ksa_expand_slots": (_int, [_vp, ctypes.c_longlong] + [_int] * 5 + [ctypes.c_longlong, _int, _int, _vp, _int]
                         + [_vp] * 3 + [ctypes.c_longlong, _int, _vp]),
    "ksa_copy_rows": (_int, [_vp] * 4 + [_int] * 6 + [_i64p] * 2 + [_vp]),
    "ksa_pre_attention": (_int, [_vp] * 10 + [_int] * 6 + [_i64p] * 7 + [_vp, _int, ctypes.c_float, _vp]),
    "ksa_pre_attention_partials": (_int, [_vp, _int] + [_vp] * 7 + [_int] * 6 + [_i64p] * 4
                                   + [_vp, _int, ctypes.c_float, _vp]),
    "ksa_add_rmsnorm": (_int, [_vp] * 5 + [ctypes.c_longlong, _int] + [ctypes.c_longlong] * 4
                        + [_int, ctypes.c_float, _vp]),
    "ksa_embed_rmsnorm": (_int, [_vp, ctypes.c_longlong, ctypes.c_longlong] + [_vp] * 4 + [_int, _int, _vp, _int, _int]
                          + [_vp, _vp, _int, ctypes.c_float, _vp]),
    "ksa_add_rmsnorm_partials": (_int, [_vp, _int] + [_vp] * 4 + [_int, _int] + [ctypes.c_longlong] * 3
                                 + [_int, ctypes.c_float, _vp]),
    "ksa_silu_mul": (_int, [_vp] * 3 + [ctypes.c_longlong, _int] + [ctypes.c_longlong] * 3 + [_int, _vp]),
    "ksa_argmax_rows": (_int, [_vp, _vp, _int, _int, ctypes.c_longlong, _int, _vp]),
    "ksa_silu_mul_partials": (_int, [_vp, _int, _vp, _int, _int, ctypes.c_longlong, _int, _vp]),
    "ksa_gemm_rows_auto_splits": (_int, [_int, _int]),
    "ksa_gemm_rows_workspace_bytes": (ctypes.c_size_t, [_int, _int]),
    "ksa_tile_weights_bytes": (ctypes.c_size_t, [_int, _int]),
    "ksa_tile_weights": (_int, [_vp, _vp, _int, _int, ctypes.c_longlong, _vp]),
    "ksa_gemm_rows_splits": (_int, [_int, _int, _int]),
    "ksa_gemm_rows_partials_bytes": (ctypes.c_size_t, [_int, _int, _int]),
    "ksa_gemm_rows": (_int, [_vp] * 3 + [_int] * 3 + [ctypes.c_longlong] * 3 + [_int, _int, _vp, ctypes.c_size_t, _vp]),
    "ksa_gemm_rows_gate_up_silu": (_int, [_vp] * 3 + [_int] * 3 + [ctypes.c_longlong] * 3 + [_int, _vp]),
    "ksa_mlp_rows_down_splits": (_int, [_int, _int]),
    "ksa_mlp_rows_workspace_bytes": (ctypes.c_size_t, [_int, _int]),
    "ksa_decode_qkv_wide_splits": (_int, [_int] * 5),
    "ksa_mlp_rows_status_offset": (ctypes.c_size_t, []),
    "ksa_mlp_rows": (_int, [_vp] * 4 + [_int] * 3 + [ctypes.c_longlong] * 3 + [_int, _vp, ctypes.c_size_t, _vp]),
    "ksa_add_rmsnorm_mlp_rows": (_int, [_vp, _int] + [_vp] * 6 + [_int] * 3 + [ctypes.c_longlong] * 4
                                 + [_int, ctypes.c_float, _vp, ctypes.c_size_t, _vp]),
    "ksa_step_workspace_bytes": (ctypes.c_size_t, []),
    "ksa_step_status_offset": (ctypes.c_size_t, []),
    "ksa_decode_qkv_o_splits": (_int, [_int] * 5),
    "ksa_decode_qkv_o_pays": (_int, [_int] * 6),
    "ksa_decode_qkv_o_workspace_bytes": (ctypes.c_size_t, [_int] * 5),
    "ksa_decode_qkv_o_fwd": (_int, [_vp, _int] + [_vp] * 4 + [ctypes.c_longlong, ctypes.c_float] + [_vp] * 3 + [_int]
                             + [_vp] * 2 + [_int] * 7 + [_i64p] * 2 + [ctypes.c_float, _int, _vp, _vp, _int, _vp,
                                                                       ctypes.c_size_t, _vp, ctypes.c_size_t, _vp]),
    "ksa_decode_qkv_o_wide_fwd": (_int, [_vp, _int] + [_vp] * 4 + [ctypes.c_longlong, ctypes.c_float] + [_vp] * 3 + [_int]
                             + [_vp] * 2 + [_int] * 7 + [_i64p] * 2 + [ctypes.c_float, _int, _vp, _vp, _int, _vp,
                                                                       ctypes.c_size_t, _vp, ctypes.c_size_t, _vp]),
    "ksa_decode_qkv_o_wide_splits": (_int, [_int] * 6),
    "ksa_decode_qkv_o_wide_pays": (_int, [_int] * 6),
    "ksa_add_rmsnorm_gemm_rows_splits": (_int, [_int] * 3),
    "ksa_add_rmsnorm_gemm_rows_pays": (_int, [_int] * 4),
    "ksa_add_rmsnorm_gemm_rows": (_int, [_vp, _int] + [_vp] * 5 + [_int] * 3 + [ctypes.c_longlong] * 2
                                  + [_int, ctypes.c_float, _vp, ctypes.c_size_t, _vp]),
    "ksa_debug_norm_gemm_rows_give_up": (_int, [_vp, _int] + [_vp] * 5 + [_int] * 4 + [ctypes.c_float, _vp, ctypes.c_size_t, _vp]),
    "ksa_debug_count_visible": (ctypes.c_longlong, [ctypes.c_longlong] * 3 + [_int] * 7),
}

EXPORTS = tuple(_SIGNATURES)


class KsaError(RuntimeError):
    pass


class _GeneralWay:
    """In place of the native front, whose parts of PyTorch are not all public: takes no call, so that every one goes the
    Python way to the same entry points of the library."""
    decode = prefill = pre_attention = block_index = staticmethod(lambda *args: None)


def lib():
    global _lib, fast
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise KsaError(
                f"{LIB_PATH} is missing: build it with `python ksa_amd/build.py` "
                "(hipcc, gfx950); ksa_amd has no other execution path")
        L = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in _SIGNATURES.items():
            fn = getattr(L, name)
            fn.restype = res
            fn.argtypes = args
        try:
            from . import _fast
            _fast.bind(check, *[ctypes.cast(getattr(L, n), ctypes.c_void_p).value for n in _FAST])
            fast = _fast
        except (ImportError, TypeError) as e:   # (TypeError: a build with other entry points)
            warnings.warn(f"ksa_amd/_fast.so is missing or was built for another PyTorch: the same kernels are called from Python, "
                          f"small calls take some 10 us longer.  Build it with `python ksa_amd/build.py` ({e})", RuntimeWarning)
            fast = _GeneralWay
        _lib = L
    return _lib


def check(code: int, what: str):
    if code != 0:
        msg = lib().ksa_error_string(code).decode()
        raise KsaError(f"{what}: {msg} (code {code})")


_I64x3 = ctypes.c_int64 * 3


def strides3(t, dims):
    """int64[3] of element strides of tensor `t` along the three named dims."""
    s = t.stride()
    return _I64x3(s[dims[0]], s[dims[1]], s[dims[2]])


def _private(*names):
    """These private functions of torch, or None where one of them is missing: its next release may have renamed it,
    and a CPU-only build has no `_cuda_*`.  What uses them then takes the public way."""
    try:
        return [functools.reduce(getattr, n.split("."), torch) for n in names]
    except AttributeError:
        return None


_GPU = _private("_C._cuda_getDevice", "_C._cuda_getCurrentRawStream")
# each false or None where nobody records, traces or transforms
_WATCHERS = _private("_C._len_torch_dispatch_stack", "_C._len_torch_function_stack",
                     "_C._functorch.peek_interpreter_stack", "_C._get_tracing_state", "autograd._profiler_enabled")


def stream_ptr(device) -> int:
    """Handle of the current stream of a GPU (asked for at every call: 0.1 us where a Stream object takes 1.5)."""
    if _GPU is None:
        return torch.cuda.current_stream(device).cuda_stream
    return _GPU[1](_GPU[0]() if device.index is None else device.index)


_HERE_ALREADY = contextlib.nullcontext()


def on_device(device):
    """Context in which `device` is the current GPU; nothing to enter (and 2 us of host time less) where it
    is that already."""
    if device.index is None or (_GPU is not None and device.index == _GPU[0]()):
        return _HERE_ALREADY
    return torch.cuda.device(device)


def direct(*tensors) -> bool:
    """Whether an operator's kernels may be called without the dispatcher (10 us of host time per call, as much
    as a small launch takes on the GPU): plain tensors, and nobody compiles, traces, records, profiles (the operator's
    name belongs into the trace) or transforms.
    (Inside `torch.func` transforms a tensor may be a wrapper of the plain type that has no storage, and a view
    with its negative bit set holds other values than its memory: the dispatcher unwraps the first, slice by
    slice, and writes out the second.  It does the same for wrappers and all-zero tensors without memory that are met
    outside of a transform.)"""
    if _WATCHERS is None or torch.compiler.is_compiling():
        return False
    modes, functions, transform, trace, profiler = _WATCHERS
    if modes() or functions() or transform() is not None or trace() is not None or profiler():
        return False
    for t in tensors:
        if t is not None and (type(t) is not torch.Tensor or (t.requires_grad and torch.is_grad_enabled())
                              or t.is_neg() or not t.data_ptr()):
            return False
    return True
