"""Test helpers: seeded inputs, the oracle on device tensors, error metrics.

Inputs follow the benchmark configurations: fp16 drawn i.i.d. N(0,1) (times an
optional factor) from a seeded generator on the CPU, then copied to the device.
"""

from __future__ import annotations

import numpy as np
import torch

from oracle import attention as orc

FWD_ATOL = 2e-3      # forward: max |O - O_ref| against the fp32/fp64 closed form
GRAD_RTOL = 1e-2     # backward: max |g - g_ref| / max |g_ref| per gradient


def randn(shape, seed, scale=1.0, device="cuda"):
    g = torch.Generator().manual_seed(seed)
    x = (torch.randn(shape, generator=g, dtype=torch.float32) * scale).half()
    return x.to(device) if device is not None else x


def np64(t: torch.Tensor) -> np.ndarray:
    return t.detach().float().cpu().numpy().astype(np.float64)


def max_abs(a, b) -> float:
    a = a.detach().float().cpu() if isinstance(a, torch.Tensor) else torch.as_tensor(a).float()
    b = b.detach().float().cpu() if isinstance(b, torch.Tensor) else torch.as_tensor(b).float()
    return float((a - b).abs().max()) if a.numel() else 0.0


def rel_err(g, ref) -> float:
    """max |g - ref| / max |ref| (0 if ref is identically zero and g matches)."""
    g = g.detach().float().cpu() if isinstance(g, torch.Tensor) else torch.as_tensor(g).float()
    ref = ref.detach().float().cpu() if isinstance(ref, torch.Tensor) else torch.as_tensor(ref).float()
    den = float(ref.abs().max()) if ref.numel() else 0.0
    num = float((g - ref).abs().max()) if g.numel() else 0.0
    return num / den if den > 0 else num


def oracle_fwd(q, k, v, scale, causal):
    o, lse = orc.attention_fwd(np64(q), np64(k), np64(v), scale, causal)
    return torch.from_numpy(o), torch.from_numpy(lse)


def oracle_bwd(q, k, v, do, scale, causal):
    dq, dk, dv = orc.attention_bwd(np64(q), np64(k), np64(v), np64(do), scale, causal)
    return torch.from_numpy(dq), torch.from_numpy(dk), torch.from_numpy(dv)


def cu_from_lens(lens, device="cuda"):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + int(n))
    return torch.tensor(cu, dtype=torch.int32, device=device)


def _c_call(fn, tensors, mid, strides, scale, causal, workspace):
    """One call of a C entry point of the library on the current stream, on operands as they are."""
    import ctypes
    from flash_attn_legacy import hip_ext
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    rc = fn(*[p(t) for t in tensors], *mid, *[(ctypes.c_int64 * 3)(*s) for s in strides], ctypes.c_float(scale),
            int(causal), p(workspace), workspace.numel(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    if rc:
        raise RuntimeError(f"status {rc}: {hip_ext._lib.fal_last_error().decode()}")


def c_backward(do, q, k, v, o, lse, scale, causal, workspace_bytes=None, nq=None):
    """fal_bwd with a workspace of `workspace_bytes` (fal_bwd_workspace_size's when None); the
    gradients start out as NaN.  `nq`: query rows, if not all of q's."""
    from flash_attn_legacy import hip_ext
    lib = hip_ext._lib
    (B, Hq, Nq, d), (_, Hkv, Nk, _) = q.shape, k.shape
    nq = Nq if nq is None else nq
    if workspace_bytes is None:
        workspace_bytes = lib.fal_bwd_workspace_size(B, Hq, nq, d)
    grads = [torch.full(s, float("nan"), dtype=q.dtype, device=q.device)
             for s in ((B, Hq, Nq, d), (B, Hkv, Nk, d), (B, Hkv, Nk, d))]
    ws = torch.empty(max(workspace_bytes, 1), dtype=torch.uint8, device=q.device)
    _c_call(lib.fal_bwd_bf16 if q.dtype == torch.bfloat16 else lib.fal_bwd, (do, q, k, v, o, lse, *grads),
            (B, Hq, Hkv, nq, Nk, d), [t.stride()[:3] for t in (do, q, k, v, o, *grads)], scale, causal, ws)
    return grads


def c_backward_varlen(do, q, k, v, o, lse, cu_q, cu_k, max_q, max_k, scale, causal, total_q=None):
    """fal_bwd_varlen, as c_backward."""
    from flash_attn_legacy import hip_ext
    lib = hip_ext._lib
    (rows_q, Hq, d), (tk, Hkv, _), seqs = q.shape, k.shape, cu_q.numel() - 1
    tq = rows_q if total_q is None else total_q
    grads = [torch.full(s, float("nan"), dtype=q.dtype, device=q.device)
             for s in ((rows_q, Hq, d), (tk, Hkv, d), (tk, Hkv, d))]
    ws = torch.empty(lib.fal_bwd_varlen_workspace_size(seqs, tq, tk, Hq, d), dtype=torch.uint8, device=q.device)
    _c_call(lib.fal_bwd_varlen_bf16 if q.dtype == torch.bfloat16 else lib.fal_bwd_varlen,
            (do, q, k, v, o, lse, *grads, cu_q, cu_k), (seqs, tq, tk, Hq, Hkv, d, max_q, max_k),
            [(0, t.stride(1), t.stride(0)) for t in (do, q, k, v, o, *grads)], scale, causal, ws)
    return grads
