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


@pytest.mark.parametrize("T,Hq,Hkv", [(70, 4, 1), (130, 4, 2), (300, 8, 2)])
def test_prompt_attention_of_infinite_values_and_scores(cuda_device, T, Hq, Hkv):
    """As in fp32: an infinite value makes its dim infinite for the queries
    that attend to it (NaN where both infinities meet), a NaN NaN, and leaves
    the other dims alone; keys whose scores are -inf drop out, also a whole
    block of 64 of them."""
    from ecf8_amd.llm_kernels import packed_kv, prompt_attention

    gen = torch.Generator(device=cuda_device).manual_seed(T)

    def rand(*shape):
        return torch.randn(shape, generator=gen, device=cuda_device).to(torch.bfloat16)

    q, kc, vc = rand(1, Hq, T, 128), rand(1, Hkv, T, 128), rand(1, Hkv, T, 128)
    work = packed_kv(1, Hkv, T, cuda_device)
    out = torch.empty(T, Hq * 128, dtype=torch.bfloat16, device=cuda_device)

    def check(rows, v, skip=()):
        prompt_attention(q, kc, v, T, work, out, Hq)
        got = out.double().view(T, Hq, 128).transpose(0, 1)[None, :, rows]
        want = _causal64(q, kc, v.nan_to_num(0, 0, 0))[:, :, rows]
        dims = [d for d in range(128) if d not in skip]
        bound = want.abs() * 2.0 ** -8 * 1.01 + float(v.nan_to_num(0, 0, 0).abs().max()) * 2.0 ** -16
        assert bool(((got - want).abs() <= bound)[..., dims].all())
        return got

    v = vc.clone()
    inf = math.inf
    v[..., 5, 3], v[..., 66, 40], v[..., 7, 100], v[..., 9, 77] = inf, -inf, inf, math.nan
    v[..., 68, 100] = -inf
    got = check(slice(68, T), v, (3, 40, 77, 100))
    assert bool((got[..., 3] == inf).all()) and bool((got[..., 40] == -inf).all())
    assert bool(got[..., 77].isnan().all()) and bool(got[..., 100].isnan().all())
    q[..., 0] = q[..., 0].abs() + 0.1
    kc[..., :64, 0] = -inf
    check(slice(64, T), vc)
    kc[..., 64:, :] = rand(1, Hkv, T - 64, 128)
    kc[..., 10, 0] = 0.5  # one key of the block remains
    check(slice(10, T), vc)


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


def _dit_reference(streams, heads, cos, sin, tail):
    """Float64 restatement of dit_kernels.joint_attention."""
    qs, ks, vs = [], [], []
    for t, nq, nk in streams:
        q, k, v = t.double().unflatten(2, (3, heads, 128)).permute(2, 0, 3, 1, 4)

        def norm(x, w):
            return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * w.weight.double()

        qs.append(norm(q, nq))
        ks.append(norm(k, nk))
        vs.append(v)

    def rope(x):
        x0, x1 = x[..., 0::2], x[..., 1::2]
        c, s = cos.double(), sin.double()
        return torch.stack([x0 * c - x1 * s, x0 * s + x1 * c], -1).flatten(-2)

    q, k, v = rope(torch.cat(qs, 2)), rope(torch.cat(ks, 2)), torch.cat(vs, 2)
    o = torch.softmax(q @ k.transpose(-1, -2).contiguous() / math.sqrt(128), -1) @ v
    o = o.transpose(1, 2).flatten(2)
    if tail is not None:
        x = tail.double()
        g = 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))
        o = torch.cat([o, g], -1)
    return o


@pytest.mark.parametrize("B,tokens,heads,tail", [
    (1, (1,), 1, 0), (1, (31, 32), 8, 0), (2, (5, 59), 2, 0), (1, (64,), 3, 8), (1, (65,), 8, 520),
    (2, (127,), 2, 264), (1, (1, 127), 1, 0), (1, (128, 1), 16, 0), (3, (200,), 4, 1024),
    # over 256 workgroups of 128 queries: the kernel of 256 queries
    (1, (1,), 264, 0), (1, (64,), 264, 8), (1, (65,), 257, 0), (1, (129,), 136, 0),
    (2, (31, 225), 72, 0), (1, (257,), 96, 0), (1, (200, 313), 66, 0)])
def test_dit_joint_attention_matches_fp64(cuda_device, B, tokens, heads, tail):
    """One stream (a strided slice of a wider projection, with a GELU tail)
    and two, at the edges of the 32-token, 64-key and 128-query tiles.
    Against fp64, relative L2: q, k and the probabilities are rounded to
    bf16 (2^-8 largest, 2^-9.8 rms), the output again: 4 * 2^-9.8."""
    from ecf8_amd import dit_kernels as DK
    from ecf8_amd.dit import _Norm

    gen = torch.Generator(device=cuda_device).manual_seed(sum(tokens) * 10 + heads)

    def rand(*shape):
        return torch.randn(shape, generator=gen, device=cuda_device).to(torch.bfloat16)

    C, streams, last = heads * 128, [], None
    for n in tokens:
        y = rand(B, n, 3 * C + tail)
        norms = [_Norm(128).to(cuda_device) for _ in range(2)]
        for m in norms:
            m.weight.data.copy_(1 + 0.2 * rand(128).float())
        streams.append((y[..., : 3 * C], *norms))
        last = y[..., 3 * C:] if tail else None
    T = sum(tokens)
    angle = torch.rand(1, 1, T, 64, generator=gen, device=cuda_device) * 6.28
    cos, sin = torch.cos(angle), torch.sin(angle)
    got = DK.joint_attention(streams, heads, cos, sin, tail=last)
    assert got.shape == (B, T, C + tail) and got.dtype == torch.bfloat16
    want = _dit_reference(streams, heads, cos, sin, last)
    for part in (slice(0, C), slice(C, C + tail)):
        if want[..., part].numel():
            err = (got[..., part].double() - want[..., part]).norm() / want[..., part].norm()
            assert float(err) <= 4 * 2.0 ** -9.8, float(err)


@pytest.mark.parametrize("heads", [2, 96])  # one and two waves a SIMD
@pytest.mark.parametrize("along,rises", [
    ((.1, .1, .45, .45, .45, .45), {2: 8}), ((.1, .1, .1, .1, .1, .5), {5: 8}),
    ((.1, .1, .29, .29, .29, .29), {2: 5}), ((.05, .2, .35, .55, .75, .95), {1: 3, 2: 3, 3: 5, 5: 5}),
    ((.1, .5, .1, .1, .9, .1), {1: 8, 4: 8})])
def test_dit_joint_attention_rescales_where_maxima_rise(cuda_device, heads, along, rises):
    """Row maxima (base-2 units) that rise by more than the 8 at which sums
    are rescaled, in a middle block of 64 keys and in the partial last one,
    by less than that, and step by step; for half of the queries of a wave
    only (the others point the other way).  The values of the first two
    blocks are 1000 times as large, so that what the rescale leaves of them
    counts.  Against fp64 on the same bf16-rounded q and k, relative L2: the
    probabilities and the output are rounded to bf16, 2^-9.8 rms each."""
    from ecf8_amd import dit_kernels as DK
    from ecf8_amd.dit import _Norm

    T, C = 5 * 64 + 17, heads * 128
    gen = torch.Generator(device=cuda_device).manual_seed(int(100 * sum(along)) + heads)

    def rand(*shape):
        return torch.randn(shape, generator=gen, device=cuda_device)

    u = rand(heads, 128)
    u = u / u.norm(dim=-1, keepdim=True) * math.sqrt(128)
    sign = torch.where(torch.arange(T, device=cuda_device) % 3 == 1, -1.0, 1.0)[:, None, None]
    a = torch.tensor(along, device=cuda_device).repeat_interleave(64)[:T, None, None]
    q = sign * u + 0.02 * rand(T, heads, 128)
    across = rand(T, heads, 128)
    across = across - (across * u).sum(-1, keepdim=True) / 128 * u
    across = across / across.norm(dim=-1, keepdim=True) * math.sqrt(128)
    k = a * u + (1 - a * a).sqrt() * across
    v = rand(T, heads, 128)
    v[:128] *= 1000
    y = torch.stack([q, k, v], 1).to(torch.bfloat16).reshape(1, T, 3 * C)
    norms = [_Norm(128).to(cuda_device).requires_grad_(False) for _ in range(2)]
    for m in norms:
        m.weight.data.fill_(1.5)
    cos = torch.ones(1, 1, T, 64, device=cuda_device)
    got = DK.joint_attention([(y, *norms)], heads, cos, torch.zeros_like(cos))

    q, k, v = y[0].double().unflatten(1, (3, heads, 128)).permute(1, 2, 0, 3)

    def norm(x, scale):
        x = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * 1.5
        return (x * scale).float().to(torch.bfloat16).double()

    s = norm(q, DK.Q_SCALE) @ norm(k, 1.0).transpose(-1, -2).contiguous()
    tops = torch.stack([b.amax(-1) for b in s.split(64, -1)], -1)[:, sign[:, 0, 0] > 0]
    for b, least in rises.items():
        rise = tops[..., b] - tops[..., :b].amax(-1)
        assert float(rise.min()) > least and (least >= 8 or float(rise.max()) < 8)
    want = (torch.softmax(s * math.log(2), -1) @ v).transpose(0, 1).reshape(T, C)
    for rows in (sign[:, 0, 0] > 0, sign[:, 0, 0] < 0):
        err = (got[0][rows].double() - want[rows]).norm() / want[rows].norm()
        assert float(err) <= 3 * 2.0 ** -9.8, float(err)


def test_dit_joint_attention_leaves_odd_layouts(cuda_device):
    """An expanded norm weight and a tail with overlapping rows run in torch."""
    from ecf8_amd import dit_kernels as DK
    from ecf8_amd.dit import _Norm

    y = torch.randn(1, 4, 3 * 128, device=cuda_device).to(torch.bfloat16)
    norms = [_Norm(128).to(cuda_device).requires_grad_(False) for _ in range(2)]
    cos = torch.ones(1, 1, 4, 64, device=cuda_device)
    tail = y.reshape(-1)[:16].expand(1, 4, 16)
    assert DK.joint_attention([(y, *norms)], 1, cos, cos, tail=tail) is None
    norms[0].weight = torch.nn.Parameter(norms[0].weight[:1].expand(128), requires_grad=False)
    assert DK.joint_attention([(y, *norms)], 1, cos, cos) is None


@pytest.mark.parametrize("B,T,C", [(1, 1, 8), (2, 3, 2048), (1, 5, 2056), (2, 2, 4096), (1, 3, 8192)])
def test_dit_elementwise_matches_torch(cuda_device, B, T, C):
    """LayerNorm modulation (fp32, one bf16 rounding: at most one ulp from
    torch's) and gated add (the same two roundings: bit-identical)."""
    import torch.nn.functional as F

    from ecf8_amd import dit_kernels as DK

    gen = torch.Generator(device=cuda_device).manual_seed(C)

    def rand(*shape):
        return torch.randn(shape, generator=gen, device=cuda_device).to(torch.bfloat16)

    x, y, emb = rand(B, T, C) + 0.5, rand(B, T, C), rand(B, 6 * C)
    shift, scale, gate = emb.chunk(6, dim=-1)[1:4]
    want = F.layer_norm(x.float(), (C,), eps=1e-6) * (1 + scale.float()[:, None])
    want = (want + shift.float()[:, None])
    got = DK.modulate(x, shift, scale)
    assert bool(((got.float() - want).abs() <= want.abs() * 2.0 ** -8 * 1.01 + 1e-5).all())
    assert torch.equal(DK.gated_add(x, gate, y), x + gate[:, None] * y)


@pytest.mark.parametrize("B", [1, 2])
@pytest.mark.parametrize("kind", ["single", "double"])
def test_dit_blocks_agree_with_the_torch_path(cuda_device, monkeypatch, kind, B):
    """A block's forward through the kernels against the same forward in
    torch: bf16 roundings at the same places, scores kept in fp32 instead of
    bf16 (2 % of the block's update), and the update added to x and rounded
    to bf16 up to twice, each rounding 2^-9.8 of x rms on either side: 2 *
    sqrt(2) * 2^-9.8 < 2^-8 of the output's norm.  Also what the kernels leave
    to torch: autograd, transposed inputs, fp16 autocast, hooks on a norm."""
    from ecf8_amd import dit_kernels as DK
    from ecf8_amd.dit import FluxConfig, random_pipeline

    cfg = FluxConfig(hidden=256, heads=2, mlp=512, double=1, single=1, txt_dim=128, pooled_dim=128)
    pipe, _ = random_pipeline(cfg, cuda_device, seed=5)
    gen = torch.Generator(device=cuda_device).manual_seed(B)

    def rand(*shape):
        return torch.randn(shape, generator=gen, device=cuda_device).to(torch.bfloat16)

    img, txt, emb = rand(B, 35, 256), rand(B, 7, 256), rand(B, 256)
    cos, sin = pipe.dit.rope_tables(7, 5, 7, cuda_device)
    blk, args = ((pipe.dit.blocks[0], (img, txt, emb)) if kind == "double"
                 else (pipe.dit.single_blocks[0], (torch.cat([txt, img], 1), emb)))
    calls = []
    monkeypatch.setattr(DK, "_launch", lambda *a, _f=DK._launch: (calls.append(a[1]), _f(*a))[1])

    def run(*a):
        calls.clear()
        out = blk(*a, cos, sin)
        return out if isinstance(out, tuple) else (out,)

    with torch.no_grad():
        fused = run(*args)
        assert "ecf8_packed_attention" in calls and "ecf8_dit_modulate" in calls
        with monkeypatch.context() as mp:
            mp.setattr(DK, "_untracked", lambda: False)
            plain = run(*args)
        assert not calls
        for a, b, x in zip(fused, plain, args):
            diff, update = (a.double() - b.double()).norm(), (b.double() - x.double()).norm()
            assert float(diff) <= 0.02 * float(update) + 2.0 ** -8 * float(b.double().norm())
        turned = [t.transpose(1, 2).contiguous().transpose(1, 2) if t.dim() == 3 else t for t in args]
        for a, b in zip(run(*turned), plain):
            assert float((a.double() - b.double()).norm() / b.double().norm()) <= 0.02
        with torch.autocast("cuda", dtype=torch.float16):
            run(*args)
        assert not calls
        norm = blk.attn.norm_k_a if kind == "double" else blk.norm_k_a
        seen = []
        handle = norm.register_forward_hook(lambda *_: seen.append(1))
        run(*args)
        handle.remove()
        assert seen and "ecf8_packed_attention" not in calls
    leaf = args[0].clone().requires_grad_()
    run(leaf, *args[1:])[0].float().sum().backward()
    assert "ecf8_packed_attention" not in calls and bool(torch.isfinite(leaf.grad).all())


def test_prompt_attention_leaves_no_workspace(cuda_device):
    """A prompt's packed keys and values go back to the allocator: nothing
    of their size stays with the runner."""
    from types import SimpleNamespace

    from ecf8_amd.llm import _GreedyRunner

    B, T, Hkv, Hq = 2, 512, 8, 32
    r = _GreedyRunner()
    r.B, r.dev, r.cfg = B, cuda_device, SimpleNamespace(heads=Hq, kv_heads=Hkv)
    r.q = torch.randn(B * Hq * T * 128, device=cuda_device).to(torch.bfloat16)
    r.kc = [torch.randn(B, Hkv, T, 128, device=cuda_device).to(torch.bfloat16)]
    r.vc = [torch.randn(B, Hkv, T, 128, device=cuda_device).to(torch.bfloat16)]
    r.attn = torch.empty(B * T, Hq * 128, dtype=torch.bfloat16, device=cuda_device)
    before = torch.cuda.memory_allocated(cuda_device)
    r._prefill_attention(0, T)
    assert torch.cuda.memory_allocated(cuda_device) == before
