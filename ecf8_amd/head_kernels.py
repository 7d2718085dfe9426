"""Python wrappers of the ends of a decode step (include/ecf8_head.h): the
bf16 linear of a few rows, the greedy next token and its embedding."""

from __future__ import annotations

import torch
import torch.nn.functional as F

from ._lib import ECF8Error, check, lib
from .guards import takes, untracked
from .llm_kernels import _need

MAX_ROWS, MAX_K = 16, 4096


def _launch(x, w, b):
    M, N = x.shape[0], w.shape[0]
    out = torch.empty(M, N, dtype=torch.bfloat16, device=x.device)
    with torch.cuda.device(x.device):
        check(lib().ecf8_bf16_linear16(x.data_ptr(), x.stride(0), M, w.shape[1], w.data_ptr(), N,
                                       None if b is None else b.data_ptr(), out.data_ptr(), N,
                                       torch.cuda.current_stream(x.device).cuda_stream),
              "ecf8_bf16_linear16")
    return out


class _SmallLinear(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, b):
        ctx.save_for_backward(x, w)
        return _launch(x, w, b)

    @staticmethod
    def backward(ctx, g):
        x, w = ctx.saved_tensors
        need = ctx.needs_input_grad
        return (g @ w if need[0] else None, g.t() @ x if need[1] else None,
                g.sum(0) if need[2] else None)


def small_linear(x, w, b=None):
    """F.linear(x, w, b); for a few rows of bf16 CUDA tensors ([M, K], M <=
    16) through the HIP kernel, otherwise the library's."""
    every = (x, w) if b is None else (x, w, b)
    if (x.dim() != 2 or w.dim() != 2 or not 1 <= x.shape[0] <= MAX_ROWS or x.stride(1) != 1
            or x.stride(0) % 8 or (x.shape[0] > 1 and x.stride(0) < x.shape[1])
            or not w.is_contiguous() or w.shape[1] != x.shape[1] or w.shape[1] % 32
            or w.shape[1] > MAX_K or w.shape[0] % 16
            or (b is not None and (tuple(b.shape) != (w.shape[0],) or not b.is_contiguous()))
            or not untracked() or not takes(every, grad=True)):
        return F.linear(x, w, b)
    if torch.is_grad_enabled() and any(t.requires_grad for t in every):
        return _SmallLinear.apply(x, w, b)
    return _launch(x, w, b)


def greedy_work(B: int, device) -> torch.Tensor:
    """Work buffer of greedy_emit."""
    n = lib().ecf8_greedy_work_bytes(B)
    if n < 0:
        raise ECF8Error("bad batch size")
    return torch.empty(n // 8, dtype=torch.int64, device=device)


def refusal_flag() -> torch.Tensor:
    """A flag in pinned host memory for ``refused=`` below: zero until a
    kernel refuses a call's values, which the host may look up at any time."""
    return torch.zeros(1, dtype=torch.int32, device="cpu", pin_memory=torch.cuda.is_available())


def _flag_ptr(refused):
    if refused is None:
        return None
    if refused.dtype != torch.int32 or not (refused.is_cuda or refused.is_pinned()):
        raise ECF8Error("refused must be int32 in pinned host or device memory")
    return refused.data_ptr()


def greedy_emit(logits, work, tokens, next_token, step, pos=None, advance: int = 0, refused=None):
    """argmax of each row of ``logits`` (bf16 [B, V]) -> next_token[b] and
    tokens[b, step[0]]; then step += 1 and pos += advance.  A step outside
    the token buffer writes no token and sets ``refused``."""
    dev = logits.device
    _need(logits, torch.bfloat16, "logits", dev)
    for t, n in ((tokens, "tokens"), (next_token, "next_token"), (step, "step"), (work, "work")):
        _need(t, torch.int64, n, dev)
    if advance:
        _need(pos, torch.int32, "pos", dev)
    B, V = logits.shape
    if tokens.dim() != 2 or tokens.shape[0] < B or next_token.numel() < B or step.numel() < 1:
        raise ECF8Error("tokens, next_token or step too small")
    with torch.cuda.device(dev):
        check(lib().ecf8_greedy_emit_checked(
            logits.data_ptr(), logits.stride(0), B, V, work.data_ptr(), work.numel() * 8,
            tokens.data_ptr(), tokens.shape[1], next_token.data_ptr(), step.data_ptr(),
            pos.data_ptr() if advance else None, advance, _flag_ptr(refused),
            torch.cuda.current_stream(dev).cuda_stream), "ecf8_greedy_emit")


def embed_rows(token, table, out, refused=None):
    """out fp32 [>= B, H] = float(table[token]) for int64 tokens [B]; a token
    outside the table writes zeros and sets ``refused``."""
    dev = out.device
    _need(token, torch.int64, "token", dev)
    _need(table, torch.bfloat16, "table", dev)
    _need(out, torch.float32, "out", dev)
    B, (V, H) = token.numel(), table.shape
    if out.dim() != 2 or out.shape[1] != H or out.shape[0] < B:
        raise ECF8Error("out does not fit the embedded rows")
    with torch.cuda.device(dev):
        check(lib().ecf8_embed_rows_checked(
            token.data_ptr(), B, table.data_ptr(), V, H, out.data_ptr(), _flag_ptr(refused),
            torch.cuda.current_stream(dev).cuda_stream), "ecf8_embed_rows")
