"""The prompt kernels of the session's prefill branch (``csrc/prefill.hip``).

``causal_attention`` takes the attention of a whole prompt where
``prefill_attention`` has no mask, ``token_scores`` the scores of
``compute_prefill_scores``.  Each returns None, launching nothing, for
inputs it does not take; the caller then runs the PyTorch form.
"""
from __future__ import annotations

import ctypes

import torch
from torch import Tensor
from torch.autograd import forward_ad
from torch.utils._python_dispatch import _get_current_dispatch_mode

from .. import _lib


def _plain(*tensors: Tensor) -> bool:
    """GPU tensors that nothing traces, transforms or differentiates: the
    kernels write their results behind autograd's back.  To be asked before
    anything else of the tensors, which may be a symbolic tracer's."""
    if torch.compiler.is_compiling() or any(type(t) is not Tensor for t in tensors):
        return False
    if torch._C._get_tracing_state() is not None or _get_current_dispatch_mode() is not None \
            or forward_ad._current_level >= 0 or torch._C._functorch.peek_interpreter_stack() is not None or torch._C._len_torch_function_stack() > 0:
        return False
    if torch.is_autocast_enabled("cuda") and tensors[0].dtype != torch.get_autocast_dtype("cuda"):
        return False  # the PyTorch form computes in, and returns, autocast's type
    grad = torch.is_grad_enabled()
    return all(t.is_cuda and t.device == tensors[0].device and not (grad and t.requires_grad) for t in tensors)


def _rows_ok(*tensors: Tensor) -> bool:
    """[B, H, S, D] with contiguous, 16-byte aligned rows."""
    for t in tensors:
        per = 16 // t.element_size()
        if t.stride(3) != 1 or t.data_ptr() % 16 or any(t.stride(i) < 0 or t.stride(i) % per for i in range(3)):
            return False
    return True


def causal_attention(q: Tensor, k: Tensor, v: Tensor, scaling: float) -> Tensor | None:
    """Causal attention [B, H, S, D] of equally long q, k, v (bf16 / f16,
    head_dim 64 or 128), the result with q's strides, as SDPA's fused
    kernels return it."""
    if not (_plain(q, k, v) and q.dim() == 4 and q.shape == k.shape == v.shape and q.dtype == k.dtype == v.dtype
            and q.dtype in (torch.bfloat16, torch.float16) and q.shape[3] in (64, 128) and q.numel() > 0
            and scaling > 0):
        return None
    out = torch.empty_like(q)
    if not _rows_ok(q, k, v, out) or max(t.stride(2) for t in (q, k, v, out)) > 1 << 22:
        return None
    B, H, S, D = q.shape
    strides = (ctypes.c_int64 * 12)(*(t.stride(i) for t in (q, k, v, out) for i in range(3)))
    with torch.cuda.device(q.device):
        _lib.check(_lib.lib().wnw_prefill_attn(
            _lib.ptr(q), _lib.ptr(k), _lib.ptr(v), B, H, H, S, D, strides, float(scaling), _lib.dtype_code(q.dtype),
            _lib.ptr(out), _lib.stream_of(q.device)), "prefill_attn")
    return out


def token_scores(q: Tensor, k: Tensor, attention_mask: Tensor | None, audio_starts: list[int], audio_ends: list[int],
                 class_a_heads: list[int], kv_heads: list[int], group: int, last: bool,
                 scaling: float) -> tuple[list, list] | None:
    """Prompt token scores of one layer in two launches
    (``wnw_prefill_scores``): per sample the class-A heads' row (None
    without class-A heads) and one row per entry of ``kv_heads``.
    ``attention_mask``: additive [B, 1, S, S], or None for causal."""
    m = attention_mask
    if not _plain(*((q, k) if m is None else (q, k, m))):
        return None
    if not (q.dim() == k.dim() == 4 and q.dtype == k.dtype and q.dtype in _lib._TORCH_DTYPES
            and q.shape[0] == k.shape[0] and q.shape[2:] == k.shape[2:] and q.shape[3] in (64, 128, 256)
            and q.shape[1] == k.shape[1] * group and q.numel() > 0):
        return None
    B, _, S, D = q.shape
    if len(audio_starts) != B or len(audio_ends) != B or max(B, len(class_a_heads), len(kv_heads)) > 64 or \
            any(not (0 <= a < e <= S) for a, e in zip(audio_starts, audio_ends)) or \
            any(not 0 <= h < q.shape[1] for h in class_a_heads) or any(not 0 <= h < k.shape[1] for h in kv_heads):
        return None
    if m is not None and not (m.dtype in _lib._TORCH_DTYPES and m.shape == (B, 1, S, S) and m.stride(3) == 1):
        return None
    if not _rows_ok(q, k):
        return None
    dev = q.device
    width = max(e - a for a, e in zip(audio_starts, audio_ends))
    most = max(len(class_a_heads), group * (1 if last else S - min(audio_ends)))
    items = len(kv_heads) + (1 if class_a_heads else 0)
    out_a = torch.empty(B, width, dtype=torch.float32, device=dev) if class_a_heads else None
    out_h = torch.empty(B, len(kv_heads), width, dtype=torch.float32, device=dev)
    dt = _lib.dtype_code(q.dtype)
    i32 = lambda x: (ctypes.c_int32 * max(len(x), 1))(*x)  # noqa: E731
    strides = (ctypes.c_int64 * 8)(*(t.stride(i) for t in (q, k) for i in range(3)),
                                   *((0, 0) if m is None else (m.stride(0), m.stride(2))))
    with torch.cuda.device(dev):
        need = int(_lib.lib().wnw_prefill_scores_workspace_bytes(B, items, S, D, most, dt))
        ws = torch.empty(need, dtype=torch.uint8, device=dev)
        _lib.check(_lib.lib().wnw_prefill_scores(
            _lib.ptr(q), _lib.ptr(k), _lib.ptr(m), strides, B, q.shape[1], k.shape[1], S, D, i32(audio_starts),
            i32(audio_ends), i32(class_a_heads), len(class_a_heads), i32(kv_heads), len(kv_heads), 1 if last else 0,
            float(scaling), dt, dt if m is None else _lib.dtype_code(m.dtype), width, most, _lib.ptr(out_a),
            _lib.ptr(out_h), _lib.ptr(ws), need, _lib.stream_of(dev)), "prefill_scores")
    n = [e - a for a, e in zip(audio_starts, audio_ends)]
    return ([out_a[b, :n[b]] if class_a_heads else None for b in range(B)],
            [[out_h[b, i, :n[b]] for i in range(len(kv_heads))] for b in range(B)])
