"""Binding of libfal_hip.so -- the drop-in for the reference's compiled
extension module ``flash_attn_legacy_cuda`` (csrc/flash_attn_legacy.cpp:294-310).

It exposes the reference's three functions with the same arguments, outputs and
error behaviour (``RuntimeError`` with the library's message):

* ``forward(Q, K, V, softmax_scale, is_causal=False) -> [O, L]``
* ``forward_varlen(Q, K, V, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k,
  softmax_scale, is_causal=False) -> [O, L]``
* ``backward(dO, Q, K, V, O, L, softmax_scale, is_causal=False) -> [dQ, dK, dV]``

plus two entry points the reference does not have:

* ``backward_varlen(...)`` -- one launch for all packed sequences;
* ``decode(q, k_cache, v_cache, cache_seqlens, softmax_scale, ...)`` -- split-K
  KV-cache decode.

Outputs and workspaces are allocated with torch on the input's device; the library itself
never allocates.  Work is enqueued on the current torch stream.  Both steps are native
(``_fal_torch``, csrc/fal_torch.cpp); ctypes loads the library, so that
``FLASH_ATTN_LEGACY_LIB`` can name another build of it.  There is no fallback: if either
shared library is missing, importing this module raises ``ImportError``.
"""

from __future__ import annotations

import ctypes
import os
from typing import List, Optional

import torch

try:
    from . import _fal_torch as _native
except ImportError as e:
    raise ImportError(f"flash_attn_legacy native binding (_fal_torch.so) not loadable: {e}. "
                      "Build it with: python flash-attention-legacy_amd/build.py") from e

_LIB_NAME = "libfal_hip.so"
# FLASH_ATTN_LEGACY_LIB selects another build of the same library (e.g. a tuning variant).
_LIB_PATH = os.environ.get("FLASH_ATTN_LEGACY_LIB") or os.path.join(
    os.path.dirname(os.path.abspath(__file__)), _LIB_NAME)

_VP = ctypes.c_void_p
_I64 = ctypes.c_int64
_F32 = ctypes.c_float
_INT = ctypes.c_int
_SZ = ctypes.c_size_t
_STR = ctypes.c_void_p   # int64[3] stride triples


def _load() -> ctypes.CDLL:
    if not os.path.exists(_LIB_PATH):
        raise ImportError(
            f"flash_attn_legacy HIP library not found at {_LIB_PATH}. "
            "Build it with: python flash-attention-legacy_amd/build.py"
        )
    lib = ctypes.CDLL(_LIB_PATH)
    sig = {
        "fal_last_error": (ctypes.c_char_p, []),
        "fal_version": (ctypes.c_char_p, []),
        "fal_device_supported": (_INT, [_INT]),
        "fal_fwd_workspace_size": (_SZ, [_I64] * 5 + [_INT]),
        "fal_fwd": (_INT, [_VP] * 5 + [_I64] * 6 + [_STR] * 4 + [_F32, _INT, _VP, _SZ, _VP]),
        "fal_fwd_varlen_workspace_size": (_SZ, [_I64] * 4),
        "fal_fwd_varlen": (_INT, [_VP] * 7 + [_I64] * 8 + [_STR] * 4 + [_F32, _INT, _VP, _SZ, _VP]),
        "fal_bwd_workspace_size": (_SZ, [_I64] * 4),
        "fal_bwd_workspace_best": (_SZ, [_I64] * 6 + [_INT]),
        "fal_bwd": (_INT, [_VP] * 9 + [_I64] * 6 + [_STR] * 8 + [_F32, _INT, _VP, _SZ, _VP]),
        "fal_bwd_varlen_workspace_size": (_SZ, [_I64] * 5),
        "fal_bwd_varlen": (_INT, [_VP] * 11 + [_I64] * 8 + [_STR] * 8 + [_F32, _INT, _VP, _SZ, _VP]),
        "fal_decode_workspace_size": (_SZ, [_I64] * 5),
        "fal_decode": (_INT, [_VP] * 5 + [_I64, _VP, _VP] + [_I64] * 5 + [_STR] * 4 + [_F32, _VP, _SZ, _VP]),
        "fal_decode_noalloc": (_INT, [_VP] * 5 + [_I64, _VP, _VP] + [_I64] * 5 + [_STR] * 4 + [_F32, _VP]),
    }
    for name in ("fal_fwd", "fal_fwd_varlen", "fal_bwd", "fal_bwd_varlen", "fal_decode"):
        sig[name + "_bf16"] = sig[name]   # bf16 forms: same arguments
    for name, (res, args) in sig.items():
        fn = getattr(lib, name)
        fn.restype = res
        fn.argtypes = args
    return lib


_lib = _load()

# Exported names, for introspection and tests.
SYMBOLS = (
    "fal_last_error", "fal_version", "fal_device_supported",
    "fal_fwd_workspace_size", "fal_fwd", "fal_fwd_varlen_workspace_size", "fal_fwd_varlen",
    "fal_bwd_workspace_size", "fal_bwd_workspace_best", "fal_bwd", "fal_bwd_varlen_workspace_size", "fal_bwd_varlen",
    "fal_decode_workspace_size", "fal_decode",
    "fal_fwd_bf16", "fal_fwd_varlen_bf16", "fal_bwd_bf16", "fal_bwd_varlen_bf16", "fal_decode_bf16",
    "fal_decode_noalloc",
)


def library_path() -> str:
    return _LIB_PATH


def version() -> str:
    return _lib.fal_version().decode()


def device_supported(device: int = 0) -> bool:
    return bool(_lib.fal_device_supported(int(device)))


# The tensor side of each call (checks, outputs, workspace, launch on the current stream) is
# native; it calls the library that is loaded above.
_native.bind({name: ctypes.cast(getattr(_lib, name), ctypes.c_void_p).value for name in SYMBOLS})

_HEAD_AXIS = {"bshd": 2, "bhsd": 1}


# ---------------------------------------------------------------------------
# Reference-compatible entry points
# ---------------------------------------------------------------------------

def forward(Q: torch.Tensor, K: torch.Tensor, V: torch.Tensor, softmax_scale: float,
            is_causal: bool = False) -> List[torch.Tensor]:
    """[O, L] for Q [B,Hq,N,d], K/V [B,Hkv,Nk,d]; L is [B,Hq,N] fp32 natural-log LSE.
    Checks of ``flash_attn_forward`` (csrc/flash_attn_legacy.cpp:48-60)."""
    return _native.forward(Q, K, V, float(softmax_scale), bool(is_causal))


def forward_varlen(Q, K, V, cu_seqlens_q, cu_seqlens_k, max_seqlen_q: int, max_seqlen_k: int,
                   softmax_scale: float, is_causal: bool = False) -> List[torch.Tensor]:
    """[O, L] for packed Q [total_q,Hq,d], K/V [total_k,Hkv,d]; L is [total_q,Hq].
    Checks of ``flash_attn_forward_varlen`` (csrc/flash_attn_legacy.cpp:201-217).
    The (sequence, tile) schedule is built on the device: no host synchronisation."""
    return _native.forward_varlen(Q, K, V, cu_seqlens_q, cu_seqlens_k, int(max_seqlen_q), int(max_seqlen_k),
                                  float(softmax_scale), bool(is_causal))


def backward(dO, Q, K, V, O, L, softmax_scale: float, is_causal: bool = False) -> List[torch.Tensor]:
    """[dQ, dK, dV] from the saved forward (O, L).  Checks of ``flash_attn_backward``
    (csrc/flash_attn_legacy.cpp:115-120); dQ has Q's shape, dK/dV have K/V's."""
    return _native.backward(dO, Q, K, V, O, L, float(softmax_scale), bool(is_causal))


# ---------------------------------------------------------------------------
# Entry points without a reference counterpart
# ---------------------------------------------------------------------------

def backward_varlen(dO, Q, K, V, O, L, cu_seqlens_q, cu_seqlens_k, max_seqlen_q: int, max_seqlen_k: int,
                    softmax_scale: float, is_causal: bool = False) -> List[torch.Tensor]:
    """[dQ, dK, dV] for packed sequences in one launch.  Same results as the reference's
    per-sequence loop (flash_attn_legacy/flash_attn.py:133-157): dK/dV rows outside every
    segment are zero."""
    return _native.backward_varlen(dO, Q, K, V, O, L, cu_seqlens_q, cu_seqlens_k, int(max_seqlen_q), int(max_seqlen_k),
                                   float(softmax_scale), bool(is_causal))


def decode(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, cache_seqlens: torch.Tensor,
           softmax_scale: float, mask_bias: Optional[torch.Tensor] = None, cache_layout: str = "bshd",
           return_lse: bool = False):
    """Split-K decode.  q [B,Hq,d] (one token per sequence); caches [B,S,Hkv,d]
    (``cache_layout="bshd"``) or [B,Hkv,S,d] (``"bhsd"``); cache_seqlens int32 [B];
    mask_bias optional fp32 [B,S] additive mask.  Returns O [B,Hq,d] (and L [B,Hq])."""
    axis = _HEAD_AXIS.get(cache_layout)
    if axis is None:
        raise RuntimeError(f"unknown cache_layout {cache_layout!r}")
    res = _native.decode(q, k_cache, v_cache, cache_seqlens, float(softmax_scale), mask_bias, axis, bool(return_lse))
    return tuple(res) if return_lse else res[0]
