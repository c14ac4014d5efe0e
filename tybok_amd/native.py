"""Binding of ``libtybok_hip.so`` (the C ABI declared in ``include/tybok_hip.h``): :func:`lib` through ctypes, for the entry
points that a program calls while it prepares, and :func:`calls`, an extension module on torch tensors, for the ones that launch.

Both are loaded from ``tybok_amd/_lib/``; there is no fallback: if one is missing or an
entry point fails, a ``RuntimeError`` is raised (the reference's native helpers raise instead
of exiting too: tybok/policies/fastwam/kernels/coop_grid.h:20-27).
"""

from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import os
import sysconfig
from ctypes import c_char_p, c_float, c_int, c_longlong, c_size_t, c_void_p

_LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_lib", "libtybok_hip.so")
_lib: ctypes.CDLL | None = None
_calls = None

# name -> (restype, argtypes); mirrors include/tybok_hip.h one to one
SIGNATURES: dict[str, tuple] = {
    "tk_version": (c_int, []),
    "tk_last_error": (c_char_p, []),
    "tk_device_cus": (c_int, []),
    "tk_workspace_bytes": (c_size_t, []),
    "tk_workspace_init": (c_int, [c_void_p, c_size_t, c_void_p]),
    "tk_fp8w_packed_bytes": (c_size_t, [c_int, c_int]),
    "tk_pack_fp8_weight": (c_int, [c_void_p, c_void_p, c_int, c_int, c_void_p]),
    "tk_pack_fp8_gate_up": (c_int, [c_void_p, c_void_p, c_void_p, c_int, c_int, c_void_p]),
    "tk_fp8w_gemm": (
        c_int,
        [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_int, c_int, c_void_p, c_int, c_int, c_int,
         c_int, c_void_p, c_size_t, c_void_p],
    ),  # fmt: skip
    "tk_fp8w_gemm_static": (
        c_int,
        [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_int, c_int, c_void_p, c_int, c_int, c_int,
         c_int, c_void_p],
    ),  # fmt: skip
    "tk_static_scratch_bytes": (c_size_t, []),
    "tk_fp8w_gated_ffn": (
        c_int,
        [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_int, c_int,
         c_void_p, c_int, c_int, c_int, c_int, c_void_p, c_size_t, c_void_p],
    ),  # fmt: skip
    "tk_fp8w_norm_gated_ffn": (
        c_int,
        [c_void_p, c_int, c_void_p, c_float, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
         c_int, c_void_p, c_int, c_int, c_void_p, c_int, c_int, c_int, c_int, c_void_p, c_size_t, c_void_p],
    ),  # fmt: skip
    "tk_set_ffn_fusion": (c_int, [c_int]),
    "tk_set_handoff_spin": (c_int, [c_int]),
    "tk_workspace_handoff_error_offset": (c_size_t, []),
    "tk_quant_act_rows": (c_int, [c_void_p, c_int, c_void_p, c_int, c_void_p, c_int, c_int, c_int, c_void_p]),
    "tk_w8a8_gemm": (
        c_int,
        [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int,
         c_void_p, c_size_t, c_void_p],
    ),  # fmt: skip
    "tk_w8a8_gated_ffn": (
        c_int,
        [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_int, c_int,
         c_int, c_int, c_int, c_int, c_int, c_void_p, c_size_t, c_void_p],
    ),  # fmt: skip
    "tk_w8a8_ffn_layout": (c_int, [c_int, c_int, c_int, c_void_p, c_void_p, c_void_p]),
    "tk_bf16w_packed_bytes": (c_size_t, [c_int, c_int]),
    "tk_pack_bf16_weight": (c_int, [c_void_p, c_void_p, c_int, c_int, c_int, c_void_p]),
    "tk_bf16w_linear": (
        c_int,
        [c_void_p, c_int, c_int, c_void_p, c_void_p, c_float, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int,
         c_int, c_int, c_void_p, c_int, c_int, c_void_p, c_int, c_void_p, c_int, c_int, c_void_p, c_int, c_int, c_int,
         c_int, c_void_p, c_size_t, c_void_p],
    ),  # fmt: skip
    "tk_bf16w_dense": (
        c_int,
        [c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p, c_int, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int,
         c_int, c_void_p, c_size_t, c_void_p],
    ),  # fmt: skip
    "tk_f16w_dense": (
        c_int,
        [c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p, c_int, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int,
         c_int, c_void_p, c_size_t, c_void_p],
    ),  # fmt: skip
    "tk_bf16w_dense_rope": (c_int, [c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int,
                                    c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_void_p, c_size_t, c_void_p]),
    "tk_bf16w_dense_vt": (c_int, [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_int, c_int, c_int, c_longlong, c_int, c_int, c_int,
                                  c_int, c_int, c_int, c_void_p, c_size_t, c_void_p]),
    "tk_prefix_meta": (c_int, [c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_void_p, c_void_p, c_void_p, c_void_p]),
    "tk_patchify_images": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_float, c_float, c_void_p, c_void_p]),
    "tk_patchify_images_f32": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_float, c_float, c_void_p, c_void_p]),
    "tk_layer_norm_f16": (c_int, [c_void_p, c_int, c_void_p, c_void_p, c_float, c_void_p, c_int, c_int, c_int, c_void_p]),
    "tk_add_layer_norm_f16": (
        c_int,
        [c_void_p, c_int, c_void_p, c_int, c_void_p, c_int, c_void_p, c_void_p, c_float, c_void_p, c_int, c_int, c_int, c_void_p],
    ),
    "tk_attn_prepare_kv": (
        c_int,
        [c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_int,
         c_void_p],
    ),  # fmt: skip
    "tk_expert_tail": (
        c_int,
        [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_float, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_float,
         c_int, c_int, c_int, c_void_p],
    ),  # fmt: skip
    "tk_expert_tail_embed": (
        c_int,
        [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_float, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_float,
         c_int, c_int, c_int, c_void_p, c_void_p, c_int, c_int, c_void_p, c_int, c_int, c_void_p],
    ),  # fmt: skip
    "tk_layer_norm": (c_int, [c_void_p, c_int, c_int, c_void_p, c_void_p, c_int, c_float, c_void_p, c_int, c_int, c_int, c_void_p]),
    "tk_expert_kv_project": (
        c_int,
        [c_void_p, c_void_p, c_int, c_int, c_int, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p],
    ),
    "tk_expert_kv_project_layers": (
        c_int,
        [c_int, c_void_p, c_void_p, c_int, c_int, c_int, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p],
    ),
    "tk_expert_cross_attn_fused": (
        c_int,
        [c_void_p, c_int, c_void_p, c_float, c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_int, c_int,
         c_void_p, c_void_p, c_int, c_int, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_void_p],
    ),  # fmt: skip
    "tk_batched_attn": (
        c_int,
        [c_void_p, c_longlong, c_int, c_int, c_void_p, c_longlong, c_int, c_int, c_void_p, c_longlong, c_int, c_int,
         c_void_p, c_longlong, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_float, c_void_p, c_size_t, c_void_p],
    ),  # fmt: skip
    "tk_batched_transpose_v": (
        c_int,
        [c_void_p, c_longlong, c_int, c_int, c_void_p, c_longlong, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_void_p],
    ),  # fmt: skip
    "tk_add_layer_norm": (
        c_int,
        [c_void_p, c_int, c_int, c_void_p, c_int, c_void_p, c_int, c_void_p, c_void_p, c_int, c_float, c_void_p, c_int, c_int, c_int, c_void_p],
    ),  # fmt: skip
    "tk_prefix_rows": (
        c_int,
        [c_void_p, c_int, c_int, c_float, c_void_p, c_void_p, c_int, c_int, c_float, c_void_p, c_int, c_void_p, c_int, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_void_p],
    ),  # fmt: skip
    "tk_add_layer_norm_rows": (
        c_int,
        [c_void_p, c_int, c_int, c_void_p, c_int, c_void_p, c_int, c_void_p, c_void_p, c_int, c_float, c_void_p, c_int, c_void_p, c_int, c_int, c_void_p],
    ),  # fmt: skip
    "tk_rms_norm_rows": (c_int, [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_float, c_void_p, c_int, c_int, c_int, c_void_p]),
    "tk_rope_rows": (c_int, [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_void_p]),
    "tk_expert_attn": (
        c_int,
        [c_void_p, c_int, c_int, c_void_p, c_void_p, c_int, c_int, c_void_p, c_void_p, c_int, c_int, c_void_p, c_int,
         c_int, c_void_p, c_int, c_int, c_void_p, c_void_p, c_int, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int,
         c_int, c_int, c_int, c_void_p, c_size_t, c_void_p],
    ),  # fmt: skip
    "tk_sv_denoise_xchg_bytes": (c_size_t, [c_int]),
    "tk_sv_denoise_layer_bytes": (c_size_t, []),
    "tk_sv_denoise_pack": (c_int, [c_void_p, c_int, c_void_p, c_size_t, c_void_p]),
    "tk_sv_denoise": (c_int, [c_void_p, c_void_p]),
    "tk_pi_denoise_xchg_bytes": (c_size_t, []),
    "tk_pi_denoise_layer_bytes": (c_size_t, []),
    "tk_pi_denoise_mod_floats": (c_size_t, []),
    "tk_pi_denoise": (c_int, [c_void_p, c_void_p]),
    "tk_debug_decode_fp8": (c_int, [c_void_p, c_void_p]),
    "tk_debug_stream_read": (c_int, [c_void_p, c_size_t, c_int, c_void_p, c_void_p]),
    "tk_debug_many_rows_gemm": (
        c_int,
        [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_int, c_int, c_void_p]
        + [c_int] * 6 + [c_void_p, c_size_t, c_void_p],
    ),  # fmt: skip
    "tk_debug_w8a8_tile": (c_int, [c_int] * 5),
    "tk_debug_linear_blocks": (c_int, [c_int] * 4),
    "tk_debug_fp8w_gemm_cut": (c_int, [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_void_p]),
}

SV_MAX_LAYERS = 20


class SvWeights(ctypes.Structure):
    """``tk_sv_weights``"""

    _fields_ = [*((n, c_void_p) for n in ("wqkv", "wo", "wgu", "wd", "sg", "su", "sd", "norm_in", "norm_post")), ("cross", c_int)]


class SvCache(ctypes.Structure):
    """``tk_sv_cache``"""

    _fields_ = [*((n, c_void_p) for n in ("k", "k_lo", "vt", "vt_lo")), *((n, c_int) for n in ("k_sl", "k_sh", "vt_sh", "vt_sd"))]


class SvDenoiseArgs(ctypes.Structure):
    """``tk_sv_denoise_args``"""

    _fields_ = [
        *((n, c_int) for n in ("layers", "steps", "M", "P")),
        ("cross_mask", ctypes.c_uint),
        *((n, c_float) for n in ("dt", "eps")),
        *((n, c_void_p) for n in ("x0", "out", "pad", "pos", "pos0", "rope_cos", "rope_sin")),
        *((n, c_int) for n in ("positions", "polls")),
        *((n, c_void_p) for n in ("emb_w", "emb_b", "time_w", "time_b", "act_w", "act_b", "blob", "xchg")),
        ("xchg_bytes", c_size_t),
        ("cache", SvCache * SV_MAX_LAYERS),
    ]


PI_MAX_LAYERS = 24


class PiCache(ctypes.Structure):
    """``tk_pi_cache``"""

    _fields_ = [*((n, c_void_p) for n in ("k", "vt")), *((n, c_int) for n in ("k_sl", "vt_sd"))]


class PiDenoiseArgs(ctypes.Structure):
    """``tk_pi_denoise_args``"""

    _fields_ = [
        *((n, c_int) for n in ("layers", "steps", "M", "P")),
        *((n, c_float) for n in ("dt", "eps")),
        *((n, c_void_p) for n in ("x0", "out", "pad", "pos", "rope_cos", "rope_sin")),
        *((n, c_int) for n in ("positions", "polls")),
        *((n, c_void_p) for n in ("emb_w", "emb_b", "act_w", "mods", "blob", "xchg")),
        ("xchg_bytes", c_size_t),
        ("cache", PiCache * PI_MAX_LAYERS),
    ]


def library_path() -> str:
    return _LIB_PATH


def lib() -> ctypes.CDLL:
    """The loaded library; raises ``RuntimeError`` when it has not been built."""
    global _lib
    if _lib is None:
        if not os.path.exists(_LIB_PATH):
            raise RuntimeError(
                f"{_LIB_PATH} is missing: build it with `python -m tybok_amd.csrc.build` "
                "(there is no CPU or torch fallback for the HIP kernels)"
            )
        handle = ctypes.CDLL(_LIB_PATH)
        for name, (restype, argtypes) in SIGNATURES.items():
            fn = getattr(handle, name)
            fn.restype = restype
            fn.argtypes = argtypes
        _lib = handle
    return _lib


def check(rc: int, what: str) -> None:
    if rc != 0:
        msg = lib().tk_last_error()
        raise RuntimeError(f"{what} failed ({rc}): {msg.decode() if msg else 'unknown error'}")


def calls_path() -> str:
    """Where the extension module of this Python and this torch lies.  It is compiled against the headers of both, and neither keeps
    the layout of what they describe between versions; so both are in its name, and a build for others is not found."""
    import torch

    return os.path.join(os.path.dirname(_LIB_PATH), f"tk_calls.{sysconfig.get_config_var('SOABI')}.torch-{torch.__version__}.so")


def calls():
    """The extension module of the launching entry points (``csrc/tk_calls.cpp``): ``calls().tk_name(...)`` takes tensors for
    pointers, launches on torch's current stream (the entry's last argument, not passed) and raises like :func:`check`."""
    global _calls
    if _calls is None:
        path = calls_path()  # (imports torch: its libraries have to be in the process)
        lib()
        if not os.path.exists(path):
            raise RuntimeError(f"{path} is missing (one is built for each Python and torch): build it with `python -m tybok_amd.csrc.build`")
        loader = importlib.machinery.ExtensionFileLoader("tk_calls", path)
        module = importlib.util.module_from_spec(importlib.util.spec_from_file_location("tk_calls", path, loader=loader))
        loader.exec_module(module)
        _calls = module
    return _calls
