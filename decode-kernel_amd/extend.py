"""Extend (prefill) attention over a token pool on the HIP kernel (dk_extend_attention).

`extend_attention` is the kernel call behind SplitKVHipBackend.forward_extend; `takes` says
whether a call is one that the kernel reads as it lies. Calls that it does not take (host
tensors, other types or head sizes, rows that are not 16-byte aligned, gradients, tracing)
stay on the backend's PyTorch path.
"""
from __future__ import annotations

import ctypes
import math
from typing import Optional, Sequence

import torch

import attention
import dk_lib

_I32_MAX = 2 ** 31 - 1024


def _aligned(t: torch.Tensor) -> bool:
    """Unit last stride, the other strides and the data multiples of 16 bytes."""
    es = t.element_size()
    return t.stride(-1) == 1 and t.data_ptr() % 16 == 0 and \
        all(s >= 0 and s * es % 16 == 0 for s in t.stride()[:-1])


def _plain(*tensors: torch.Tensor) -> bool:
    """Ordinary tensors outside tracing, transforms and gradients: what a call that hands
    out raw pointers may take."""
    if torch._C._len_torch_dispatch_stack() > 0 or torch._C._get_tracing_state() is not None or \
            torch.autograd.forward_ad._current_level >= 0:
        return False
    grad = torch.is_grad_enabled()
    return all(type(t) is torch.Tensor and not (grad and t.requires_grad) and
               not torch._C._functorch.is_functorch_wrapped_tensor(t) and
               not t.is_neg() and not t.is_conj() for t in tensors)


def takes(q, k_pool, v_pool, req_to_token, rows: Sequence[int], new_lens: Sequence[int],
          all_lens: Sequence[int], scale: float, logit_cap: Optional[float],
          k_scale: float, v_scale: float, sinks: Optional[torch.Tensor]) -> bool:
    """Whether extend_attention runs this call as the PyTorch path would. The sizes that the
    PyTorch path refuses (a row or length outside the map, more new tokens than q rows or
    than the request holds) are not taken, so that they are refused there."""
    ts = (q, k_pool, v_pool, req_to_token) + (() if sinks is None else (sinks,))
    if not all(isinstance(t, torch.Tensor) for t in ts) or not _plain(*ts):
        return False
    if q.device.type != "cuda" or any(t.device != q.device for t in ts):
        return False
    if q.dtype not in (torch.float16, torch.bfloat16) or k_pool.dtype != v_pool.dtype or \
            k_pool.dtype not in (q.dtype, attention.KV_FP8):
        return False
    if q.dim() != 3 or k_pool.dim() != 3 or v_pool.shape != k_pool.shape or \
            q.shape[2] != k_pool.shape[2] or q.shape[2] not in attention.SUPPORTED_HEAD_DIMS:
        return False
    hq, hkv = q.shape[1], k_pool.shape[1]
    if hkv == 0 or hq == 0 or hq % hkv or k_pool.shape[0] == 0 or k_pool.shape[0] > _I32_MAX:
        return False
    if not (_aligned(q) and _aligned(k_pool) and _aligned(v_pool)):
        return False
    if req_to_token.dtype != torch.int32 or req_to_token.dim() != 2 or \
            req_to_token.stride(1) != 1 or req_to_token.stride(0) < req_to_token.shape[1]:
        return False
    if sinks is not None and (sinks.dtype != torch.float32 or sinks.shape != (hq,) or
                              not sinks.is_contiguous()):
        return False
    if not all(math.isfinite(x) for x in (scale * k_scale, v_scale, logit_cap or 0.0)) or \
            scale * k_scale < 1e-30 or max(k_pool.stride(0), v_pool.stride(0)) > _I32_MAX // 2:
        return False
    n_rows, width = req_to_token.shape
    return sum(new_lens) <= min(q.shape[0], _I32_MAX // hq) and \
        all(0 <= n <= t <= min(width, _I32_MAX) and -n_rows <= r < n_rows
            for r, n, t in zip(rows, new_lens, all_lens))


def extend_attention(q, k_pool, v_pool, req_to_token, rows: Sequence[int],
                     new_lens: Sequence[int], all_lens: Sequence[int], out, scale: float,
                     logit_cap: Optional[float] = None, window: Optional[int] = None,
                     k_scale: float = 1.0, v_scale: float = 1.0,
                     sinks: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Causal attention of each request's new tokens over its cached tokens (a call that
    `takes` accepts), into `out` (shaped as q, rows past the last new token untouched).

    q                  : (tokens, q_heads, head_dim), the requests' new tokens in order
    k_pool, v_pool     : (slots, kv_heads, head_dim), the new tokens already written
    req_to_token       : (rows, max_tokens) int32 slot of each request's tokens
    rows, new_lens, all_lens : host integers per request
    """
    n = len(rows)
    ints = ctypes.c_int32 * n
    n_rows = req_to_token.shape[0]
    s = dk_lib.DkExtendStrides(q.stride(0), q.stride(1), k_pool.stride(0), k_pool.stride(1),
                               v_pool.stride(0), v_pool.stride(1), out.stride(0), out.stride(1))
    kv8 = k_pool.dtype == attention.KV_FP8
    lib = dk_lib.load()
    hq, hkv, d = q.shape[1], k_pool.shape[1], q.shape[2]
    news, alls = ints(*new_lens), ints(*all_lens)
    need = lib.dk_extend_workspace_bytes(n, news, alls, hq, hkv, d, window or 0)
    ws = torch.empty(need, dtype=torch.uint8, device=q.device) if need else None
    with torch.cuda.device(q.device):
        rc = lib.dk_extend_attention(
            q.data_ptr(), k_pool.data_ptr(), v_pool.data_ptr(), req_to_token.data_ptr(),
            req_to_token.stride(0), n_rows, ints(*(r % n_rows for r in rows)), news, alls,
            out.data_ptr(), None if ws is None else ws.data_ptr(), need, n, q.shape[0], hq, hkv, d,
            k_pool.shape[0], attention._DTYPE_CODE[q.dtype],
            dk_lib.DK_KV_FP8_E4M3 if kv8 else dk_lib.DK_KV_SAME, ctypes.byref(s),
            scale * k_scale, v_scale, logit_cap or 0.0, window or 0,
            None if sinks is None else sinks.data_ptr(),
            torch.cuda.current_stream(q.device).cuda_stream)
    dk_lib.check(rc, "extend_attention")
    return out
