"""Python wrappers of the DiT block kernels (include/ecf8_attn.h): joint
attention with its head norms and rotary embedding, and the fused
elementwise passes.

Each function returns None when its kernel does not take the call, and the
caller then runs the same computation in torch: other devices, dtypes,
head dimensions, strides and alignments, tensors that autograd, forward-mode
AD, functorch or a tracer follows, tensor subclasses, dispatch modes and
autocast."""

from __future__ import annotations

import ctypes
import math

import torch

from ._lib import check, lib
from .guards import takes as _takes
from .guards import untracked as _untracked
from .llm_kernels import packed_kv

HEAD_DIM = 128
Q_SCALE = math.log2(math.e) / math.sqrt(HEAD_DIM)  # of scores that are powers of two


class _Stream(ctypes.Structure):
    _fields_ = [("qkv", ctypes.c_void_p), ("q_norm", ctypes.c_void_p), ("k_norm", ctypes.c_void_p),
                ("tokens", ctypes.c_int64), ("row_stride", ctypes.c_int64),
                ("batch_stride", ctypes.c_int64)]


def _vector(t, B, C) -> bool:
    """[B, C], columns contiguous, batches in whole 16-byte steps."""
    return tuple(t.shape) == (B, C) and t.stride(1) == 1 and t.stride(0) % 8 == 0


def _launch(dev, name, *args):
    with torch.cuda.device(dev):
        check(getattr(lib(), name)(*args, torch.cuda.current_stream(dev).cuda_stream), name)


def modulate(x, shift, scale, eps=1e-6):
    """bf16(LayerNorm(x) * (1 + scale) + shift) of x [B, T, C], or None."""
    if x.dim() != 3 or not _untracked() or not _takes((x, shift, scale)):
        return None
    B, T, C = x.shape
    if (not x.is_contiguous() or C % 8 or C > 8192 or not _vector(shift, B, C)
            or not _vector(scale, B, C)):
        return None
    out = torch.empty_like(x)
    _launch(x.device, "ecf8_dit_modulate", x.data_ptr(), B, T, C, shift.data_ptr(),
            shift.stride(0), scale.data_ptr(), scale.stride(0), eps, out.data_ptr())
    return out


def gated_add(x, gate, y):
    """x + gate[:, None] * y of x, y [B, T, C] (bf16 product), or None."""
    if x.dim() != 3 or y.shape != x.shape or not _untracked() or not _takes((x, gate, y)):
        return None
    B, T, C = x.shape
    if not x.is_contiguous() or not y.is_contiguous() or C % 8 or not _vector(gate, B, C):
        return None
    out = torch.empty_like(x)
    _launch(x.device, "ecf8_dit_gated_add", x.data_ptr(), gate.data_ptr(), gate.stride(0),
            y.data_ptr(), B, T, C, out.data_ptr())
    return out


def _qkv_rows(t, heads) -> bool:
    return (t.dim() == 3 and t.shape[2] == 3 * heads * HEAD_DIM and t.stride(2) == 1
            and t.stride(1) % 8 == 0 and t.stride(0) % 8 == 0 and t.stride(1) >= t.shape[2]
            and (t.shape[0] == 1 or t.stride(0) >= t.stride(1)))


def joint_attention(streams, heads, cos, sin, tail=None):
    """Attention over the tokens of one or two streams, in order: streams =
    [(qkv [B, T_i, 3 * heads * 128], norm_q module, norm_k module)], cos /
    sin fp32 [1, 1, T, 64].  Returns bf16 [B, T, heads * 128], or None.
    ``tail`` [B, T, m]: GELU (tanh) of it follows the heads in the result's
    columns."""
    norms = [n for _, *pair in streams for n in pair]
    if not _untracked():
        return None
    every = [s[0] for s in streams] + [n.weight for n in norms]
    if not _takes(every if tail is None else every + [tail]) or not _takes((cos, sin),
                                                                           torch.float32):
        return None
    B, T = streams[0][0].shape[0], sum(s[0].shape[1] for s in streams if s[0].dim() == 3)
    if (any(not _qkv_rows(s[0], heads) or s[0].shape[0] != B for s in streams)
            or any(tuple(n.weight.shape) != (HEAD_DIM,) or not n.weight.is_contiguous()
                   for n in norms)
            or any(tuple(t.shape) != (1, 1, T, HEAD_DIM // 2) or not t.is_contiguous()
                   or t.device != every[0].device for t in (cos, sin))):
        return None
    C, m = heads * HEAD_DIM, 0
    if tail is not None:
        m = tail.shape[-1]
        if (tuple(tail.shape) != (B, T, m) or m % 8 or tail.stride(2) != 1
                or tail.stride(1) % 8 or tail.stride(1) < m
                or (B > 1 and tail.stride(0) != T * tail.stride(1))):
            return None
    dev = every[0].device
    arr = (_Stream * len(streams))(*[
        _Stream(t.data_ptr(), q.weight.data_ptr(), k.weight.data_ptr(), t.shape[1], t.stride(1),
                t.stride(0)) for t, q, k in streams])
    q = torch.empty(B * T * C, dtype=torch.bfloat16, device=dev)
    k, v = packed_kv(B, heads, T, dev)
    out = torch.empty(B, T, C + m, dtype=torch.bfloat16, device=dev)
    _launch(dev, "ecf8_dit_qkv", arr, len(streams), B, heads, 1e-6, Q_SCALE, cos.data_ptr(),
            sin.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr())
    _launch(dev, "ecf8_packed_attention", q.data_ptr(), k.data_ptr(), v.data_ptr(), B, heads, T,
            out.data_ptr(), C + m)
    if m:
        _launch(dev, "ecf8_dit_gelu", tail.data_ptr(), tail.stride(1), B * T, m,
                out.data_ptr() + 2 * C, C + m)
    return out
