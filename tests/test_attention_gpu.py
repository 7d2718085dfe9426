"""GPU numerics of the many-query attention kernels (include/ecf8_attn.h)
against float64 restatements in torch.

Tolerance of the prompt's attention: outputs are rounded to bf16 (7 stored
mantissa bits: half an ulp is at most 2^-8 of the value); scores, softmax
and sums are fp32, whose error stays below 2^-16 of the largest value a row
averages over."""

from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _causal64(q, k, v):
    G = q.shape[1] // k.shape[1]
    k, v = (t.double().repeat_interleave(G, 1) for t in (k, v))
    s = q.double() @ k.transpose(-1, -2).contiguous() / math.sqrt(128)
    T = q.shape[2]
    s.masked_fill_(torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1), -math.inf)
    return torch.softmax(s, -1) @ v


@pytest.mark.parametrize("B,T,Hq,Hkv,Lmax", [
    (1, 1, 8, 2, 1), (2, 31, 4, 1, 40), (1, 32, 16, 2, 33), (3, 33, 3, 3, 64), (1, 63, 8, 8, 63),
    (1, 64, 4, 1, 200), (2, 65, 32, 4, 65), (1, 127, 4, 4, 128), (1, 128, 8, 1, 128),
    (1, 129, 2, 1, 300), (2, 257, 5, 1, 257)])
def test_prompt_attention_matches_fp64(cuda_device, B, T, Hq, Hkv, Lmax):
    """Query tiles, key blocks and packed tiles at their edges; the caches
    past the prompt hold NaN, which must not be read."""
    from ecf8_amd.llm_kernels import packed_kv, prompt_attention

    gen = torch.Generator(device=cuda_device).manual_seed(T * 100 + Hq)

    def rand(*shape):
        return torch.randn(shape, generator=gen, device=cuda_device).to(torch.bfloat16)

    q, kc, vc = rand(B, Hq, T, 128) * 2, rand(B, Hkv, Lmax, 128) * 2, rand(B, Hkv, Lmax, 128)
    kc[:, :, T:] = math.nan
    vc[:, :, T:] = math.nan
    out = torch.full((B * T + 1, Hq * 128), 3.0, dtype=torch.bfloat16, device=cuda_device)
    work = packed_kv(B, Hkv, T, cuda_device)
    for w in work:
        w.fill_(math.nan)
    prompt_attention(q, kc, vc, T, work, out, Hq)
    want = _causal64(q, kc[:, :, :T], vc[:, :, :T]).permute(0, 2, 1, 3).reshape(B * T, -1)
    bound = want.abs() * 2.0 ** -8 * 1.01 + float(vc[:, :, :T].abs().max()) * 2.0 ** -16
    assert bool(((out[: B * T].double() - want).abs() <= bound).all())
    assert bool((out[B * T:] == 3.0).all())


def test_prompt_attention_refuses_what_does_not_fit(cuda_device):
    from ecf8_amd._lib import ECF8Error
    from ecf8_amd.llm_kernels import packed_kv, prompt_attention

    def zeros(*shape):
        return torch.zeros(shape, dtype=torch.bfloat16, device=cuda_device)

    work = packed_kv(1, 1, 8, cuda_device)
    q, kc, out = zeros(1, 4, 8, 128), zeros(1, 1, 8, 128), zeros(8, 512)
    for bad in (dict(T=9), dict(q=zeros(1, 4, 7, 128)), dict(out=zeros(7, 512)),
                dict(work=(work[0][:64], work[1])), dict(kc=kc.float()), dict(Hq=5)):
        a = {**dict(q=q, kc=kc, T=8, work=work, out=out, Hq=4), **bad}
        with pytest.raises(ECF8Error):
            prompt_attention(a["q"], a["kc"], a["kc"], a["T"], a["work"], a["out"], a["Hq"])
