"""GPU numerics of the consumer kernels (include/ecf8_llm.h) against plain
torch fp32/fp64 restatements of the same math, and the end-to-end Qwen3-shaped
model: a model decoded from ECF8 produces exactly the tokens and logits of
the same model kept in FP8 (same kernels, bit-exact weights), eager and
graph-replayed, and its prefill logits match a torch fp32 forward of the
same architecture.

Tolerances (written per test): bf16 outputs 2^-7 relative; e4m3fn outputs
are checked after dequantization against the unquantized reference with
the format's half-ulp (2^-4 relative, plus the subnormal step) and a small
allowance for the kernels' single-precision rsqrt/exp."""

from __future__ import annotations

import math
import sys

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn


def pad16(m):
    return (m + 15) // 16 * 16


def to_tiles(x):
    from ecf8_amd.llm_kernels import to_tiles as t

    return t(x)


def from_tiles(t, R, K):
    from ecf8_amd.llm_kernels import from_tiles as f

    return f(t, R, K)


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _rand_fp8(shape, gen, dev):
    """Finite random e4m3fn bytes (0x7F / 0xFF are NaN)."""
    b = torch.randint(0, 256, shape, generator=gen, dtype=torch.int32).to(torch.uint8)
    b[(b & 0x7F) == 0x7F] = 0x7E
    return b.view(FP8).to(dev)


def _ref_quant(x):
    """The activation quantization the kernels implement, on the CPU:
    scale = amax / 448 per 1x128 group (1 if all zero), q = RNE(x / scale)."""
    x = x.float().cpu()
    M, Kd = x.shape
    g = x.view(M, Kd // 128, 128)
    amax = g.abs().amax(-1)
    s = torch.where(amax > 0, amax / 448.0, torch.ones_like(amax))
    q = (g / s[..., None]).to(FP8).view(M, Kd)
    return q, s


def _dequant(q, s):
    M, Kd = q.shape
    return (q.float().view(M, Kd // 128, 128) * s.float()[..., None]).view(M, Kd)


def _assert_fp8_close(q, s, ref, rel=2 ** -4 + 2e-3):
    """Dequantized e4m3fn vs the unquantized reference."""
    got = _dequant(q.cpu(), s.cpu())
    ref = ref.float().cpu()
    M, Kd = ref.shape
    step = (s.cpu().float()[..., None] * 2 ** -9).expand(M, Kd // 128, 128).reshape(M, Kd)
    err = (got - ref).abs()
    bound = rel * ref.abs() + step + 1e-6
    assert bool((err <= bound).all()), f"max excess {(err - bound).max().item()}"


# ------------------------------------------------------------ quantization


def test_act_quant_matches_torch_cast(cuda_device):
    from ecf8_amd.llm_kernels import act_quant

    gen = torch.Generator().manual_seed(1)
    M, Kd = 7, 8192
    x = (torch.randn(M, Kd, generator=gen) * torch.logspace(-6, 3, Kd)[torch.randperm(Kd, generator=gen)])
    x[2, 128:256] = 0.0   # an all-zero group gets scale 1
    x[3, :5] = torch.tensor([448.0, -1e-8, 3e-3, 2 ** -10, -(2 ** -7)])
    x = x.to(torch.bfloat16)
    q = torch.empty(pad16(M), Kd, dtype=FP8, device=cuda_device)  # tile layout
    s = torch.empty(M, Kd // 128, device=cuda_device)
    act_quant(x.to(cuda_device), M, q, s)
    qr, sr = _ref_quant(x)
    assert torch.equal(s.cpu(), sr)
    assert torch.equal(from_tiles(q, M, Kd).cpu().view(torch.uint8), qr.view(torch.uint8))


@pytest.mark.parametrize("Kd", [768, 2048, 4096 + 640])
def test_act_quant_rows_of_any_group_multiple(cuda_device, Kd):
    """Rows that are not a multiple of 4096 (the MoE shapes): the workgroup
    covering a row's tail writes nothing past the row -- neither the pad
    rows of the 16-row tile nor past the buffer."""
    from ecf8_amd.llm_kernels import act_quant

    gen = torch.Generator().manual_seed(Kd)
    M = 5
    x = (torch.randn(M, Kd, generator=gen) * 3).to(torch.bfloat16)
    flat = torch.full((16 * Kd + 4096,), 0x11, dtype=torch.uint8, device=cuda_device)
    q = flat[: 16 * Kd].view(FP8).view(16, Kd)
    s = torch.empty(M, Kd // 128, device=cuda_device)
    act_quant(x.to(cuda_device), M, q, s)
    qr, sr = _ref_quant(x)
    assert torch.equal(s.cpu(), sr)
    rows = from_tiles(q, 16, Kd).cpu().view(torch.uint8)
    assert torch.equal(rows[:M], qr.view(torch.uint8))
    assert bool((rows[M:] == 0x11).all())
    assert bool((flat[16 * Kd:].cpu() == 0x11).all())


@pytest.mark.parametrize("exponents", [(-126, 127), (-70, -50), (50, 70), (-20, 20)])
def test_act_quant_bytes_over_the_exponent_range(cuda_device, exponents):
    """Byte for byte the clamped cast of the fp32 quotient: groups whose
    scale is inside, outside and at the ends of the range of the short
    division, signed zeros, products that round at ties, infinities and NaN
    (clamped to 448; the sign of inf / inf is not defined)."""
    from ecf8_amd.llm_kernels import act_quant

    lo, hi = exponents
    gen = torch.Generator().manual_seed(hi)
    M, Kd = 64, 2048
    e = torch.randint(lo, hi + 1, (M, Kd // 128, 1), generator=gen).double()
    x = (1 + torch.randint(0, 128, (M, Kd // 128, 128), generator=gen) / 128) * torch.exp2(
        e - torch.randint(0, 20, (M, Kd // 128, 128), generator=gen))
    x = x * (torch.randint(0, 2, x.shape, generator=gen) * 2 - 1)
    x[0, :, ::3] = 0.0
    x[1, :, ::3] = -0.0
    x[2, ::2, 5] = float("inf")
    x[3, ::2, 7] = float("nan")
    # the largest of a group 448 x 2^n: every code and every tie is a value
    ties = torch.cat([torch.arange(1, 32) / 1024, torch.arange(17, 64) / 32, torch.arange(1, 51) * 8])
    x[4, :, 0], x[4, :, 1:1 + ties.numel() - 1] = 448 * torch.exp2(e[4, :, 0] - 8), (
        ties[:-1] * torch.exp2(e[4] - 8))
    x = x.view(M, Kd).to(torch.bfloat16)
    q = torch.empty(pad16(M), Kd, dtype=FP8, device=cuda_device)
    s = torch.empty(M, Kd // 128, device=cuda_device)
    act_quant(x.to(cuda_device), M, q, s)
    g = x.float().view(M, Kd // 128, 128)
    amax = g.abs().nan_to_num(nan=0.0, posinf=float("inf")).amax(-1)
    sr = torch.where(amax > 0, amax / 448.0, torch.ones_like(amax))
    y = g / sr[:, :, None]
    y = torch.where(y.isnan(), torch.full_like(y, 448.0).copysign(g), y.clamp(-448.0, 448.0))
    ref = y.to(FP8).view(torch.uint8).view(M, Kd)
    got = from_tiles(q, M, Kd).cpu().view(torch.uint8)
    assert torch.equal(s.cpu(), sr)
    free = (g.isinf() & sr.isinf()[:, :, None]).view(M, Kd)
    assert torch.equal(got[~free], ref[~free])
    assert bool(((got[free] & 0x7F) == 0x7E).all())


# ------------------------------------------------------------ FP8 linear


def _linear_ref(aq, a_s, segs):
    """fp64: sum_g (sum_{k in g} a*w) * a_s[m,g] * w_s[n/128,g], per segment."""
    a = aq.cpu().double()
    M, Kd = a.shape
    outs = []
    for w, ws in segs:
        wd = w.cpu().double()
        n = wd.shape[0]
        part = torch.einsum("mgk,ngk->mng", a.view(M, Kd // 128, 128), wd.view(n, Kd // 128, 128))
        scale = a_s.cpu().double()[:, None, :] * ws.cpu().double().repeat_interleave(128, 0)[None]
        outs.append((part * scale).sum(-1))
    return torch.cat(outs, dim=1)


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("M,Kd", [(1, 1024), (5, 1024), (16, 1024), (16, 8192), (3, 12288),
                                  (17, 1024), (64, 1024), (130, 1024), (300, 4096), (513, 2048)])
def test_fp8_linear_matches_fp64(cuda_device, M, Kd, layout):
    """M <= 16 runs the one-tile kernel (16 waves here: at most one
    16-column tile per CU, or K >= 8192; the 8-wave shape is checked
    below);
    larger M the LDS-tiled GEMM (256 x 128 tiles, partial row tiles at M =
    17..513).  Weights row-major (layout 0) or in the tile layout (1);
    activations always in the tile layout."""
    from ecf8_amd.llm_kernels import LinearPlan

    _say(f"[llm] fp8_linear M={M} K={Kd}")
    gen = torch.Generator().manual_seed(M * 7 + Kd)
    shapes = [256, 128, 384]
    aq = _rand_fp8((M, Kd), gen, cuda_device)
    a_s = (torch.rand(M, Kd // 128, generator=gen) * 1e-2 + 1e-4).to(cuda_device)
    segs = []
    for n in shapes:
        w = _rand_fp8((n, Kd), gen, cuda_device)
        ws = (torch.rand(n // 128, Kd // 128, generator=gen) * 1e-3 + 1e-5).to(cuda_device)
        segs.append((w, ws))
    ldo = sum(shapes) + 64
    out = torch.full((M, ldo), 7.0, dtype=torch.bfloat16, device=cuda_device)
    plan_w = [(to_tiles(w), ws, 1) if layout else (w, ws) for w, ws in segs]
    LinearPlan(plan_w, out)(to_tiles(aq), a_s, M)
    ref = _linear_ref(aq, a_s, segs)
    got = out[:, : sum(shapes)].double().cpu()
    tol = 2 ** -7 * ref.abs() + 1e-4 * ref.abs().max()
    assert bool(((got - ref).abs() <= tol).all())
    assert bool((out[:, sum(shapes):].cpu() == 7.0).all())  # columns past the segments untouched


@pytest.mark.parametrize("M", [1, 16])
def test_fp8_linear_eight_wave_shape_matches_fp64(cuda_device, M):
    """More 16-column tiles than CUs (but not the persistent K = 4096 form):
    the eight-wave kernel, q/k/v-shaped segments."""
    from ecf8_amd.llm_kernels import LinearPlan

    cus = torch.cuda.get_device_properties(cuda_device).multi_processor_count
    Kd = 1024
    shapes = [16 * cus, 512, 512]  # > cus tiles in all
    gen = torch.Generator().manual_seed(91 + M)
    aq = _rand_fp8((M, Kd), gen, cuda_device)
    a_s = (torch.rand(M, Kd // 128, generator=gen) * 1e-2 + 1e-4).to(cuda_device)
    segs = []
    for n in shapes:
        w = _rand_fp8((n, Kd), gen, cuda_device)
        ws = (torch.rand(n // 128, Kd // 128, generator=gen) * 1e-3 + 1e-5).to(cuda_device)
        segs.append((w, ws))
    out = torch.full((M, sum(shapes)), 7.0, dtype=torch.bfloat16, device=cuda_device)
    LinearPlan([(to_tiles(w), ws, 1) for w, ws in segs], out)(to_tiles(aq), a_s, M)
    ref = _linear_ref(aq, a_s, segs)
    got = out.double().cpu()
    tol = 2 ** -7 * ref.abs() + 1e-4 * ref.abs().max()
    assert bool(((got - ref).abs() <= tol).all())


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("M,shapes,Kd", [
    (17, (128,), 128), (31, (128, 256, 128), 384), (32, (4096,), 1024), (32, (4096, 128), 1152),
    (32, (12288, 384), 256), (33, (128,), 2176), (48, (4096, 256), 1024), (64, (128,), 12288),
    (64, (12416,), 256), (65, (2048, 128), 1024), (127, (2048, 128, 128), 640), (129, (2048,), 896),
    (700, (512, 128), 384), (2048, (1024,), 256), (2113, (1024,), 256), (2113, (128, 1024), 512)])
def test_fp8_linear_many_rows_either_form(cuda_device, M, shapes, Kd, layout):
    """Both forms above 16 rows, at the edges of their row blocks (32, 64,
    256) and strips (16, 32 and 64 columns in one, two and four panels),
    with fewer K groups than waves and uneven runs; the last two shapes are
    past the 512 blocks of 64 x 64 that the middle form takes on 256 CUs."""
    from ecf8_amd.llm_kernels import LinearPlan

    gen = torch.Generator().manual_seed(M * 7 + Kd)
    aq = _rand_fp8((M, Kd), gen, cuda_device)
    a_s = (torch.rand(M, Kd // 128, generator=gen) * 1e-2 + 1e-4).to(cuda_device)
    segs = [(_rand_fp8((n, Kd), gen, cuda_device),
             (torch.rand(n // 128, Kd // 128, generator=gen) * 1e-3 + 1e-5).to(cuda_device))
            for n in shapes]
    N = sum(shapes)
    out = torch.full((M + 1, N + 64), 7.0, dtype=torch.bfloat16, device=cuda_device)
    LinearPlan([(to_tiles(w), ws, 1) if layout else (w, ws) for w, ws in segs], out)(
        to_tiles(aq), a_s, M)
    a = aq.double().view(M, Kd // 128, 128) * a_s.double()[:, :, None]
    ref = torch.cat([a.view(M, Kd) @ (w.double().view(-1, 128, Kd // 128, 128)
                                      * ws.double()[:, None, :, None]).view(-1, Kd).t()
                     for w, ws in segs], 1)
    tol = 2 ** -7 * ref.abs() + 1e-4 * ref.abs().max()  # bf16 output, as above
    assert bool(((out[:M, :N].double() - ref).abs() <= tol).all())
    assert bool((out[:, N:] == 7.0).all()) and bool((out[M:] == 7.0).all())


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("shapes,Kd,pad", [
    ((4096, 1024, 1024), 4096, 0), ((4096,), 4096, 0), ((1024,), 12288, 0),
    ((128, 256, 128), 384, 2), ((512, 128), 2176, 1), ((8192,), 896, 4)])
def test_fp8_linear_rows_do_not_depend_on_the_call(cuda_device, shapes, Kd, pad, layout):
    """Above 16 rows every form adds the K groups in one order: the rows of a
    short call have the bits that they have inside a long one (tile GEMM),
    with any number of panels and row blocks, K groups that fill the waves'
    rounds or not, and row strides that take narrow stores."""
    from ecf8_amd.llm_kernels import LinearPlan

    gen = torch.Generator(device=cuda_device).manual_seed(Kd + sum(shapes))

    def fp8(n, k):
        return torch.randn(n, k, generator=gen, device=cuda_device).to(FP8)

    N = sum(shapes)
    rows = 2048 if N > 1024 else 8448  # past two 64 x 64 blocks per CU
    cus = torch.cuda.get_device_properties(cuda_device).multi_processor_count
    assert rows // 64 * (N // 64) > 2 * cus
    aq = fp8(rows, Kd)
    a_s = torch.rand(rows, Kd // 128, generator=gen, device=cuda_device) + 0.1
    segs = [(fp8(n, Kd), torch.rand(n // 128, Kd // 128, generator=gen, device=cuda_device) + 0.1)
            for n in shapes]
    out = torch.full((rows, N + pad), 7.0, dtype=torch.bfloat16, device=cuda_device)
    plan = LinearPlan([(to_tiles(w), ws, 1) if layout else (w, ws) for w, ws in segs], out)
    full = plan(to_tiles(aq), a_s, rows).clone()
    for M in (17, 32, 33, 64, 65, 135, 256, 320, 321, 512, 1000):
        out.fill_(7.0)
        plan(to_tiles(aq[:M]), a_s[:M], M)
        assert torch.equal(out[:M, :N].view(torch.int16), full[:M, :N].view(torch.int16)), M
        assert bool((out[:, N:] == 7.0).all()) and bool((out[M:] == 7.0).all()), M


@pytest.mark.parametrize("T", [17, 64, 135, 320])
def test_prompt_layer_of_one_sequence_is_that_of_a_batch(cuda_device, T):
    """A sequence's prompt pass has the same bits alone (17 to 320 rows) as
    beside others (the linears of that call through the tile GEMM): what the
    layer quantizes between its linears leaves no room for another order."""
    from ecf8_amd.llm import Qwen3Config, Qwen3ForCausalLM, Qwen3Runner
    from ecf8_amd.synth import quantize_fp8_blockwise

    cfg = Qwen3Config(layers=1, intermediate=4096, vocab=128)
    gen = torch.Generator(device=cuda_device).manual_seed(T)

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=cuda_device)

    model = Qwen3ForCausalLM(cfg).to(cuda_device)
    layer = model.model.layers[0]
    for name, (o, i, sigma) in cfg.linear_shapes().items():
        lin = layer.get_submodule(name)
        w, s = quantize_fp8_blockwise(sigma * randn(o, i))
        lin.weight, lin.weight_scale_inv = torch.nn.Parameter(w, requires_grad=False), s
    B = -(-4096 // T)
    x = randn(B * T, cfg.hidden)
    got = []
    for b in (1, B):
        r = Qwen3Runner(model, b, T, T, cuda_device)
        r.pos.zero_()
        r.res.copy_(x[: b * T])
        mlp = layer(r, 0, None, True)
        got.append([t[:n].clone() for t, n in ((mlp, T), (r.res, T), (r.kc[0], 1), (r.vc[0], 1))])
    for one, many in zip(*got):
        assert torch.equal(one, many)


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("M,extra,Kd,ldo", [
    (257, (), 128, 0), (300, (128,), 256, 0), (511, (128, 128), 896, 1), (512, (256, 128), 1152, 2),
    (1024, (384,), 128, 4), (2048, (128,), 640, 0),
])
def test_fp8_linear_wide_tiles(cuda_device, M, extra, Kd, ldo, layout):
    """256 x 256 tiles (more 256 x 128 tiles than CUs, up to as many wide
    ones): segments that end in the middle of a tile, a half-empty last one,
    1, 2 and more K groups, partial rows; row strides of 1, 2 and 4 columns
    more take stores of 2 bytes instead of 16."""
    from ecf8_amd.llm_kernels import LinearPlan

    cus = torch.cuda.get_device_properties(cuda_device).multi_processor_count
    rows = -(-M // 256)
    shapes = (128 * (cus // rows + 1), *extra)
    assert rows * sum(shapes) // 128 > cus >= rows * -(-sum(shapes) // 256)
    gen = torch.Generator().manual_seed(M + Kd)
    aq = _rand_fp8((M, Kd), gen, cuda_device)
    a_s = (torch.rand(M, Kd // 128, generator=gen) * 1e-2 + 1e-4).to(cuda_device)
    segs = [(_rand_fp8((n, Kd), gen, cuda_device),
             (torch.rand(n // 128, Kd // 128, generator=gen) * 1e-3 + 1e-5).to(cuda_device))
            for n in shapes]
    N = sum(shapes)
    out = torch.full((M + 1, N + ldo), 7.0, dtype=torch.bfloat16, device=cuda_device)
    LinearPlan([(to_tiles(w), ws, 1) if layout else (w, ws) for w, ws in segs], out)(
        to_tiles(aq), a_s, M)
    a = (aq.double().view(M, Kd // 128, 128) * a_s.double()[:, :, None]).view(M, Kd)
    ref = torch.cat([a @ (w.double().view(-1, 128, Kd // 128, 128)
                          * ws.double()[:, None, :, None]).view(-1, Kd).t() for w, ws in segs], 1)
    tol = 2 ** -7 * ref.abs() + 1e-4 * ref.abs().max()  # bf16 output, as above
    assert bool(((out[:M, :N].double() - ref).abs() <= tol).all())
    assert bool((out[:, N:] == 7.0).all()) and bool((out[M:] == 7.0).all())


def test_fp8_linear_persistent_path_matches_fp64(cuda_device):
    """More 16-column tiles than one workgroup per CU at K = 4096 (the
    gate/up shape) takes the persistent kernel that keeps the activations
    in registers and prefetches the next tile."""
    from ecf8_amd.llm_kernels import LinearPlan

    gen = torch.Generator().manual_seed(9)
    M, Kd = 16, 4096
    cus = torch.cuda.get_device_properties(cuda_device).multi_processor_count
    n = 16 * (cus + 40) // 128 * 128 + 128  # > cus tiles, a 128-multiple
    aq = _rand_fp8((M, Kd), gen, cuda_device)
    a_s = (torch.rand(M, Kd // 128, generator=gen) * 1e-2 + 1e-4).to(cuda_device)
    w = _rand_fp8((n, Kd), gen, cuda_device)
    ws = (torch.rand(n // 128, Kd // 128, generator=gen) * 1e-3 + 1e-5).to(cuda_device)
    out = torch.empty(M, n, dtype=torch.bfloat16, device=cuda_device)
    ref = _linear_ref(aq, a_s, [(w, ws)])
    LinearPlan([(w, ws)], out)(to_tiles(aq), a_s, M)
    got = out.double().cpu()
    assert bool(((got - ref).abs() <= 2 ** -7 * ref.abs() + 1e-4 * ref.abs().max()).all())
    rows_out = out.clone()
    # the same product from tile-layout weights, bit for bit
    LinearPlan([(to_tiles(w), ws, 1)], out)(to_tiles(aq), a_s, M)
    assert torch.equal(out.view(torch.int16), rows_out.view(torch.int16))


def test_fp8_linear_is_deterministic(cuda_device):
    from ecf8_amd.llm_kernels import LinearPlan

    gen = torch.Generator().manual_seed(5)
    aq = _rand_fp8((16, 4096), gen, cuda_device)
    a_s = torch.rand(16, 32, generator=gen).to(cuda_device)
    w = _rand_fp8((512, 4096), gen, cuda_device)
    ws = torch.rand(4, 32, generator=gen).to(cuda_device)
    out = torch.empty(16, 512, dtype=torch.bfloat16, device=cuda_device)
    p = LinearPlan([(w, ws)], out)
    aqt = to_tiles(aq)
    first = p(aqt, a_s, 16).clone()
    for _ in range(3):
        assert torch.equal(p(aqt, a_s, 16), first)


# ------------------------------------------------------------ row kernels


def _rms_ref(r, x, w, eps):
    r2 = r + x.float() if x is not None else r.clone()
    y = r2 * torch.rsqrt(r2.pow(2).mean(-1, keepdim=True) + eps) * w.float()
    return r2, y


@pytest.mark.parametrize("Kd", [4096, 2048])
@pytest.mark.parametrize("with_x", [False, True])
def test_rmsnorm_residual_and_outputs(cuda_device, with_x, Kd):
    from ecf8_amd.llm_kernels import rmsnorm

    gen = torch.Generator().manual_seed(3)
    M = 9
    r = torch.randn(M, Kd, generator=gen) * 3
    x = (torch.randn(M, Kd, generator=gen)).to(torch.bfloat16) if with_x else None
    w = (1 + 0.1 * torch.randn(Kd, generator=gen)).to(torch.bfloat16)
    r_ref, y_ref = _rms_ref(r, x, w, 1e-6)
    dev = cuda_device
    # bf16 output
    rd = r.to(dev)
    ob = torch.empty(M, Kd, dtype=torch.bfloat16, device=dev)
    rmsnorm(rd, w.to(dev), 1e-6, M, x=None if x is None else x.to(dev), out_bf16=ob)
    assert torch.equal(rd.cpu(), r_ref)  # one IEEE add per element
    assert torch.allclose(ob.float().cpu(), y_ref, rtol=2 ** -7, atol=1e-6)
    # fp8 output
    rd = r.to(dev)
    q = torch.empty(pad16(M), Kd, dtype=FP8, device=dev)
    s = torch.empty(M, Kd // 128, device=dev)
    rmsnorm(rd, w.to(dev), 1e-6, M, x=None if x is None else x.to(dev), out_q=q, out_scale=s)
    _assert_fp8_close(from_tiles(q, M, Kd), s, y_ref)
    # both outputs: the fp8 form is act_quant of the bf16 form, bit for bit
    rd = r.to(dev)
    ob2 = torch.empty(M, Kd, dtype=torch.bfloat16, device=dev)
    q2 = torch.empty(pad16(M), Kd, dtype=FP8, device=dev)
    s2 = torch.empty(M, Kd // 128, device=dev)
    rmsnorm(rd, w.to(dev), 1e-6, M, x=None if x is None else x.to(dev), out_q=q2, out_scale=s2,
            out_bf16=ob2)
    assert torch.equal(ob2, ob)
    qr, sr = _ref_quant(ob2)
    assert torch.equal(s2.cpu(), sr)
    assert torch.equal(from_tiles(q2, M, Kd).cpu().view(torch.uint8), qr.view(torch.uint8))


@pytest.mark.parametrize("I", [8192, 768])
def test_silu_mul_quant(cuda_device, I):
    from ecf8_amd.llm_kernels import silu_mul_quant

    gen = torch.Generator().manual_seed(4)
    M = 6
    gu = (torch.randn(M, 2 * I, generator=gen) * 4).to(torch.bfloat16)
    g, u = gu.float()[:, :I], gu.float()[:, I:]
    ref = g * torch.sigmoid(g) * u
    q = torch.empty(pad16(M), I, dtype=FP8, device=cuda_device)
    s = torch.empty(M, I // 128, device=cuda_device)
    silu_mul_quant(gu.to(cuda_device), M, q, s)
    _assert_fp8_close(from_tiles(q, M, I), s, ref)


# ------------------------------------------------------ rotary + caches


def _rope_tables(Lmax, theta=1e6):
    inv = 1.0 / (theta ** (torch.arange(0, 128, 2, dtype=torch.float64) / 128))
    ang = torch.arange(Lmax, dtype=torch.float64)[:, None] * inv[None]
    return torch.cos(ang).float(), torch.sin(ang).float()


def _qk_ref(x, w, cos, sin, eps):
    """HF Qwen3: RMSNorm over the head, then q*cos + rotate_half(q)*sin."""
    y = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w.float()
    c = torch.cat([cos, cos], -1)
    s_ = torch.cat([sin, sin], -1)
    rot = torch.cat([-y[..., 64:], y[..., :64]], -1)
    return y * c + rot * s_


def test_qk_norm_rope_writes_q_and_caches(cuda_device):
    from ecf8_amd.llm_kernels import qk_norm_rope

    gen = torch.Generator().manual_seed(6)
    B, T, Hq, Hkv, Lmax, pos0 = 3, 5, 8, 2, 32, 7
    dev = cuda_device
    qkv = torch.randn(B * T, (Hq + 2 * Hkv) * 128, generator=gen).to(torch.bfloat16)
    qn = (1 + 0.1 * torch.randn(128, generator=gen)).to(torch.bfloat16)
    kn = (1 + 0.1 * torch.randn(128, generator=gen)).to(torch.bfloat16)
    cos, sin = _rope_tables(Lmax)
    q_out = torch.zeros(B * Hq * T * 128, dtype=torch.bfloat16, device=dev)
    kc = torch.full((B, Hkv, Lmax, 128), 3.0, dtype=torch.bfloat16, device=dev)
    vc = torch.full_like(kc, 3.0)
    pos = torch.tensor([pos0], dtype=torch.int32, device=dev)
    qk_norm_rope(qkv.to(dev), B, T, Hq, Hkv, qn.to(dev), kn.to(dev), 1e-6, cos.to(dev),
                 sin.to(dev), pos, q_out, kc, vc)
    x = qkv.float().view(B, T, Hq + 2 * Hkv, 128)
    p = torch.arange(pos0, pos0 + T)
    cq, sq = cos[p][None, :, None], sin[p][None, :, None]
    q_ref = _qk_ref(x[:, :, :Hq], qn, cq, sq, 1e-6).permute(0, 2, 1, 3)
    k_ref = _qk_ref(x[:, :, Hq:Hq + Hkv], kn, cq, sq, 1e-6).permute(0, 2, 1, 3)
    v_ref = x[:, :, Hq + Hkv:].permute(0, 2, 1, 3)
    tol = dict(rtol=2 ** -7, atol=2e-2)
    assert torch.allclose(q_out.view(B, Hq, T, 128).float().cpu(), q_ref, **tol)
    assert torch.allclose(kc[:, :, pos0:pos0 + T].float().cpu(), k_ref, **tol)
    assert torch.equal(vc[:, :, pos0:pos0 + T].float().cpu(), v_ref)
    outside = torch.ones(Lmax, dtype=torch.bool)
    outside[pos0:pos0 + T] = False
    assert bool((kc[:, :, outside].cpu() == 3.0).all()) and bool((vc[:, :, outside].cpu() == 3.0).all())


# ------------------------------------------------------------ attention


@pytest.mark.parametrize("pos0,G", [(0, 4), (255, 4), (256, 4), (517, 4), (0, 8), (517, 8)])
def test_decode_attention_matches_fp32(cuda_device, pos0, G):
    """G query heads per KV head: 4 (Qwen3-8B) or 8 (Qwen3-30B-A3B)."""
    from ecf8_amd.llm_kernels import attention_work, decode_attention

    _say(f"[llm] decode_attention pos={pos0} G={G}")
    gen = torch.Generator().manual_seed(pos0)
    B, Hkv, Lmax = 3, 2, 600
    Hq = G * Hkv
    dev = cuda_device
    q = torch.randn(B, Hq, 128, generator=gen).to(torch.bfloat16)
    kc = (torch.randn(B, Hkv, Lmax, 128, generator=gen) * 2).to(torch.bfloat16)
    vc = torch.randn(B, Hkv, Lmax, 128, generator=gen).to(torch.bfloat16)
    pos = torch.tensor([pos0], dtype=torch.int32, device=dev)
    work = attention_work(B, Hq, Lmax, dev)
    oq = torch.empty(pad16(B), Hq * 128, dtype=FP8, device=dev)
    os_ = torch.empty(B, Hq, device=dev)
    ob = torch.empty(B, Hq * 128, dtype=torch.bfloat16, device=dev)
    decode_attention(q.to(dev), kc.to(dev), vc.to(dev), pos, work, oq, os_, Hq, out_bf16=ob)
    L = pos0 + 1
    k = kc[:, :, :L].float().repeat_interleave(Hq // Hkv, 1)
    v = vc[:, :, :L].float().repeat_interleave(Hq // Hkv, 1)
    sc = torch.matmul(q.float()[:, :, None], k.transpose(-1, -2).contiguous())[:, :, 0] / math.sqrt(128)
    ref = torch.matmul(torch.softmax(sc, -1)[:, :, None], v)[:, :, 0].reshape(B, Hq * 128)
    assert torch.allclose(ob.float().cpu(), ref, rtol=2 ** -7, atol=1e-4)
    _assert_fp8_close(from_tiles(oq, B, Hq * 128), os_, ref, rel=2 ** -4 + 5e-3)


@pytest.mark.parametrize("G", [4, 8])
def test_decode_attention_takes_a_v_cache_at_any_dword(cuda_device, G):
    """The values' cache may start at any multiple of 4 bytes: the same bits
    as from a 16-byte aligned one."""
    from ecf8_amd.llm_kernels import attention_work, decode_attention

    B, Hkv, Lmax = 2, 2, 300
    Hq, dev = G * Hkv, cuda_device
    gen = torch.Generator(device=dev).manual_seed(G)

    def rand(*shape):
        return torch.randn(shape, generator=gen, device=dev).to(torch.bfloat16)

    q, kc, vc = rand(B, Hq, 128), rand(B, Hkv, Lmax, 128), rand(B, Hkv, Lmax, 128)
    pos = torch.tensor([Lmax - 1], dtype=torch.int32, device=dev)
    work = attention_work(B, Hq, Lmax, dev)
    oq = torch.empty(pad16(B), Hq * 128, dtype=FP8, device=dev)
    os_, got = torch.empty(B, Hq, device=dev), []
    for at in (0, 2, 4, 6):
        v = torch.empty(vc.numel() + 8, dtype=torch.bfloat16, device=dev)[at:at + vc.numel()]
        assert v.data_ptr() % 16 == 2 * at
        v = v.view(vc.shape).copy_(vc)
        ob = torch.empty(B, Hq * 128, dtype=torch.bfloat16, device=dev)
        decode_attention(q, kc, v, pos, work, oq, os_, Hq, out_bf16=ob)
        got.append(ob)
    assert all(torch.equal(o, got[0]) for o in got)


@pytest.mark.parametrize("G", [4, 8])
@pytest.mark.parametrize("p", [0, 1, 30, 31, 32, 33, 63, 64, 223, 254, 255, 256, 287, 288, 700])
def test_fused_decode_attention_at_the_edges_of_its_splits(cuda_device, p, G):
    """Positions at the edges of a wave's 64 and a workgroup's 256; the
    caches from the new position on hold NaN, which must not reach a result.
    Against fp64 on bf16-rounded q and k (2^-8 relative for the bf16 output
    plus 2^-16 of the largest value)."""
    from ecf8_amd.llm_kernels import attention_work, decode_attention_fused

    B, Hkv, Lmax = 3, 2, 701
    Hq, dev = G * Hkv, cuda_device
    gen = torch.Generator(device=dev).manual_seed(p * 10 + G)

    def rand(*shape):
        return torch.randn(shape, generator=gen, device=dev).to(torch.bfloat16)

    qkv, kc, vc = rand(B, (Hq + 2 * Hkv) * 128), rand(B, Hkv, Lmax, 128), rand(B, Hkv, Lmax, 128)
    kc[:, :, p:] = float("nan")
    vc[:, :, p:] = float("nan")
    qn, kn = (1 + 0.1 * rand(128).float()).bfloat16(), (1 + 0.1 * rand(128).float()).bfloat16()
    cos, sin = (t.to(dev) for t in _rope_tables(Lmax))
    pos = torch.tensor([p], dtype=torch.int32, device=dev)
    out_q = torch.zeros(16, Hq * 128, dtype=torch.uint8, device=dev).view(torch.float8_e4m3fn)
    out_s, out_b = torch.zeros(B, Hq, device=dev), torch.zeros(B, Hq * 128, dtype=torch.bfloat16,
                                                               device=dev)
    old_k, old_v = kc.clone(), vc.clone()
    decode_attention_fused(qkv, B, Hq, Hkv, qn, kn, 1e-6, cos, sin, pos, kc, vc,
                           attention_work(B, Hq, Lmax, dev), out_q, out_s, out_b)
    x = qkv.double().view(B, Hq + 2 * Hkv, 128)

    def rope(t, w):
        t = t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()
        a, b = t[..., :64], t[..., 64:]
        c, s = cos[p].double(), sin[p].double()
        return torch.cat([a * c - b * s, b * c + a * s], -1)

    assert torch.equal(vc[:, :, p], qkv.view(B, -1, 128)[:, Hq + Hkv:])
    k_new = rope(x[:, Hq:Hq + Hkv], kn)
    assert torch.allclose(kc[:, :, p].double(), k_new, rtol=2 ** -7, atol=1e-6)
    keep = torch.arange(Lmax, device=dev) != p
    for new, old in ((kc, old_k), (vc, old_v)):  # nothing else is written
        assert torch.equal(new[:, :, keep].view(torch.int16), old[:, :, keep].view(torch.int16))
    q = rope(x[:, :Hq], qn).bfloat16().double()
    k = kc[:, :, :p + 1].double().repeat_interleave(G, 1)
    v = vc[:, :, :p + 1].double().repeat_interleave(G, 1)
    w = torch.softmax((q[:, :, None] * k).sum(-1) / 128 ** 0.5, -1)
    want = (w[..., None] * v).sum(2)
    # q and k are rounded to bf16 from fp32 here and from fp64 above: a
    # flipped last bit of q moves a score by up to 2^-8 of |q_i k_i|
    err = (out_b.double().view(B, Hq, 128) - want).abs()
    assert float(err.max()) <= 2.0 ** -6 * float(v.abs().max())
    assert float(err.norm() / want.norm()) <= 2.0 ** -8
    deq = from_tiles(out_q, B, Hq * 128).double().view(B, Hq, 128) * out_s.double()[..., None]
    assert float((deq - want).norm() / want.norm()) <= 2.0 ** -4


def test_wrappers_reject_bad_arguments_before_launch(cuda_device):
    """Missing outputs, short norm weights, scale buffers with too few rows
    and an empty position tensor are refused on the host; nothing is
    launched."""
    from ecf8_amd._lib import ECF8Error
    from ecf8_amd.llm_kernels import (act_quant, attention_work, decode_attention, qk_norm_rope,
                                      rmsnorm, silu_mul_quant)

    dev = cuda_device
    bf = dict(dtype=torch.bfloat16, device=dev)
    res = torch.zeros(2, 4096, device=dev)
    with pytest.raises(ECF8Error, match="out_bf16, or out_q"):
        rmsnorm(res, torch.ones(4096, **bf), 1e-6, 2)
    q8 = torch.empty(16, 4096, dtype=FP8, device=dev)  # tile layout: rows padded to 16
    with pytest.raises(ECF8Error, match="tile-layout"):
        rmsnorm(res, torch.ones(4096, **bf), 1e-6, 2, out_q=q8[:2],
                out_scale=torch.empty(2, 32, device=dev))
    for short in (torch.empty(1, 32, device=dev), torch.empty(32, device=dev)):
        with pytest.raises(ECF8Error, match="is not"):
            rmsnorm(res, torch.ones(4096, **bf), 1e-6, 2, out_q=q8, out_scale=short)
        with pytest.raises(ECF8Error, match="is not"):
            act_quant(torch.zeros(2, 4096, **bf), 2, q8, short)
        with pytest.raises(ECF8Error, match="is not"):
            silu_mul_quant(torch.zeros(2, 8192, **bf), 2, q8, short)
    B, T, Hq, Hkv, Lmax = 1, 1, 8, 2, 16
    qkv = torch.zeros(B * T, (Hq + 2 * Hkv) * 128, **bf)
    cos = torch.ones(Lmax, 64, device=dev)
    q_out = torch.zeros(B * Hq * T * 128, **bf)
    kc = torch.zeros(B, Hkv, Lmax, 128, **bf)
    vc = torch.zeros_like(kc)
    pos = torch.zeros(1, dtype=torch.int32, device=dev)
    with pytest.raises(ECF8Error, match="q_norm"):
        qk_norm_rope(qkv, B, T, Hq, Hkv, torch.ones(64, **bf), torch.ones(128, **bf), 1e-6, cos,
                     cos, pos, q_out, kc, vc)
    with pytest.raises(ECF8Error, match="pos"):
        qk_norm_rope(qkv, B, T, Hq, Hkv, torch.ones(128, **bf), torch.ones(128, **bf), 1e-6, cos,
                     cos, pos[:0], q_out, kc, vc)
    work = attention_work(B, Hq, Lmax, dev)
    oq = torch.empty(pad16(B), Hq * 128, dtype=FP8, device=dev)
    with pytest.raises(ECF8Error, match="pos"):
        decode_attention(q_out, kc, vc, pos[:0], work, oq, torch.empty(B, Hq, device=dev), Hq)


# ------------------------------------------------------------ end to end


SMALL = dict(layers=2, intermediate=4096, vocab=1024)


@pytest.fixture(scope="module")
def small_models(cuda_device):
    from ecf8_amd.llm import Qwen3Config, compress_layers, random_model

    cfg = Qwen3Config(**SMALL)
    plain, drawn = random_model(cfg, cuda_device, seed=1)
    comp, _ = random_model(cfg, cuda_device, seed=1)
    compress_layers(comp, drawn)
    return cfg, plain, comp


def _prompt(cfg, B, T):
    g = torch.Generator().manual_seed(11)
    return torch.randint(0, cfg.vocab, (B, T), generator=g)


def test_compressed_model_matches_uncompressed_exactly(small_models, cuda_device):
    from ecf8_amd.llm import Qwen3Runner
    from dfloat.run.run import TensorManager

    cfg, plain, comp = small_models
    B, T, new = 2, 16, 8
    prompt = _prompt(cfg, B, T)
    results = {}
    for name, model in (("fp8", plain), ("ecf8", comp)):
        for graph in (False, True):
            _say(f"[llm] e2e {name} graph={graph}")
            TensorManager.clear_device()
            r = Qwen3Runner(model, B, T, T + new, cuda_device)
            if graph:
                r.capture()
            toks = r.generate(prompt, new).cpu()
            last = r.logits.float().cpu()
            results[(name, graph)] = (toks, last)
    from ecf8_amd.prefetch import LayerPrefetcher

    # the default grid (2 workgroups per CU), then a quarter of a workgroup
    # per CU: most CUs without a decode workgroup, several tasks each
    for wpc in (2, 0.25):
        pf = LayerPrefetcher(comp.model.layers, cuda_device, workgroups_per_cu=wpc).install()
        for graph in (False, True):
            _say(f"[llm] e2e ecf8 prefetch wpc={wpc} graph={graph}")
            r = Qwen3Runner(comp, B, T, T + new, cuda_device)
            if graph:
                r.capture()
            for rep in range(2):  # the second run starts from the state the first left
                toks = r.generate(prompt, new).cpu()
                results[("ecf8_prefetch", wpc, graph, rep)] = (toks, r.logits.float().cpu())
            del r
        pf.uninstall()
    # re-tiled: the decode-step linears decode their weight operands
    # themselves (ECF8-T), the prompt decodes each tiled Linear first
    from ecf8_amd.llm import retile_layers

    retile_layers(comp)
    assert not hasattr(comp.model.layers[0], "encoded")
    for graph in (False, True):
        _say(f"[llm] e2e ecf8 fused graph={graph}")
        TensorManager.clear_device()
        r = Qwen3Runner(comp, B, T, T + new, cuda_device)
        if graph:
            r.capture()
        for rep in range(2):
            toks = r.generate(prompt, new).cpu()
            results[("ecf8_fused", graph, rep)] = (toks, r.logits.float().cpu())
        del r
    base_t, base_l = results[("fp8", False)]
    for key, (t, l) in results.items():
        assert torch.equal(t, base_t), key
        assert torch.equal(l, base_l), key
    assert len(set(base_t.reshape(-1).tolist())) > 1


def _torch_forward(model, prompt):
    """fp32 torch forward of the prompt with the same quantization points
    as the kernels (activations per 1x128 group before every linear)."""
    cfg = model.config
    B, T = prompt.shape
    Hq, Hkv = cfg.heads, cfg.kv_heads
    emb = model.model.embed_tokens.weight.float().cpu()
    r = emb[prompt.reshape(-1)]

    def lin(x, mod):
        q, s = _ref_quant(x)
        w = mod.weight.float().cpu()
        ws = mod.weight_scale_inv.cpu().repeat_interleave(128, 0).repeat_interleave(128, 1)
        return _dequant(q, s) @ (w * ws[: w.shape[0], : w.shape[1]]).t()

    def norm(x, w):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + cfg.eps) * w.float().cpu()

    cos, sin = _rope_tables(T, cfg.rope_theta)
    for layer in model.model.layers:
        a, m = layer.self_attn, layer.mlp
        h = norm(r, layer.input_layernorm.weight)
        q = lin(h, a.q_proj).to(torch.bfloat16).float().view(B, T, Hq, 128)
        k = lin(h, a.k_proj).to(torch.bfloat16).float().view(B, T, Hkv, 128)
        v = lin(h, a.v_proj).to(torch.bfloat16).float().view(B, T, Hkv, 128)
        # q and k are stored as bf16 after the rotary embedding
        q = _qk_ref(q, a.q_norm.weight.cpu(), cos[None, :, None], sin[None, :, None], cfg.eps)
        k = _qk_ref(k, a.k_norm.weight.cpu(), cos[None, :, None], sin[None, :, None], cfg.eps)
        q, k = q.to(torch.bfloat16).float(), k.to(torch.bfloat16).float()
        q, k, v = (t.permute(0, 2, 1, 3) for t in (q, k, v))
        k = k.repeat_interleave(Hq // Hkv, 1)
        v = v.repeat_interleave(Hq // Hkv, 1)
        s = torch.matmul(q, k.transpose(-1, -2).contiguous()) / math.sqrt(128)
        s.masked_fill_(torch.ones(T, T, dtype=torch.bool).triu(1), float("-inf"))
        o = torch.matmul(torch.softmax(s, -1), v).permute(0, 2, 1, 3).reshape(B * T, Hq * 128)
        r = r + lin(o.to(torch.bfloat16).float(), a.o_proj).to(torch.bfloat16).float()
        h = norm(r, layer.post_attention_layernorm.weight)
        g = lin(h, m.gate_proj).to(torch.bfloat16).float()
        u = lin(h, m.up_proj).to(torch.bfloat16).float()
        r = r + lin(g * torch.sigmoid(g) * u, m.down_proj).to(torch.bfloat16).float()
    h = norm(r, model.model.norm.weight).to(torch.bfloat16).float()
    last = h.view(B, T, -1)[:, -1]
    return last @ model.lm_head.weight.float().cpu().t()


def _rel(a, b):
    a, b = a.float().cpu().reshape(-1), b.float().cpu().reshape(-1)
    return ((a - b).norm() / b.norm()).item()


def _lin_deq(x_deq, mod):
    w = mod.weight.float().cpu()
    ws = mod.weight_scale_inv.cpu().repeat_interleave(128, 0).repeat_interleave(128, 1)
    return x_deq @ (w * ws[: w.shape[0], : w.shape[1]]).t()


def test_prefill_layer_stages_match_torch(small_models, cuda_device):
    """One decoder layer of the prefill, stage by stage, each stage's torch
    reference fed with the engine's own inputs to that stage: the wiring
    (norm placement, q/k/v split, head layout, GQA mapping, residual flow,
    gate/up order) is checked to bf16 rounding (relative L2 <= 1e-2; the
    inputs' fp8 codes differ from the reference quantizer's in ~0.04 % of
    elements, from single-precision rsqrt)."""
    from ecf8_amd.llm import Qwen3Runner

    cfg, plain, _ = small_models
    B, T = 2, 16
    M = B * T
    prompt = _prompt(cfg, B, T)
    r = Qwen3Runner(plain, B, T, T + 1, cuda_device)
    layer = plain.model.layers[0]
    a, m = layer.self_attn, layer.mlp
    emb = torch.nn.functional.embedding(prompt.to(cuda_device).reshape(-1),
                                        plain.model.embed_tokens.weight)
    r.res[:M].copy_(emb)
    r.pos.zero_()
    res0 = r.res[:M].float().cpu().clone()
    layer(r, 0, None, True)
    torch.cuda.synchronize()

    def norm(x, w):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + cfg.eps) * w.float().cpu()

    def lin_q(x, mod):
        q, s = _ref_quant(x)
        return _lin_deq(_dequant(q, s), mod)

    h = norm(res0, layer.input_layernorm.weight)
    qkv_ref = torch.cat([lin_q(h, a.q_proj), lin_q(h, a.k_proj), lin_q(h, a.v_proj)], 1)
    assert _rel(r.qkv[:M], qkv_ref) < 1e-2
    x = r.qkv[:M].float().cpu().view(B, T, 48, 128)
    cos, sin = _rope_tables(T, cfg.rope_theta)
    cq, sq = cos[None, :, None], sin[None, :, None]
    q_ref = _qk_ref(x[:, :, :32], a.q_norm.weight.cpu(), cq, sq, cfg.eps).permute(0, 2, 1, 3)
    k_ref = _qk_ref(x[:, :, 32:40], a.k_norm.weight.cpu(), cq, sq, cfg.eps).permute(0, 2, 1, 3)
    q = r.q[: B * 32 * T * 128].view(B, 32, T, 128)
    assert _rel(q, q_ref) < 1e-2 and _rel(r.kc[0][:, :, :T], k_ref) < 1e-2
    assert torch.equal(r.vc[0][:, :, :T].float().cpu(), x[:, :, 40:].permute(0, 2, 1, 3))
    qf, kf = q.float().cpu(), r.kc[0][:, :, :T].float().cpu().repeat_interleave(4, 1)
    vf = r.vc[0][:, :, :T].float().cpu().repeat_interleave(4, 1)
    sc = torch.matmul(qf, kf.transpose(-1, -2).contiguous()) / math.sqrt(128)
    sc.masked_fill_(torch.ones(T, T, dtype=torch.bool).triu(1), float("-inf"))
    o_ref = torch.matmul(torch.softmax(sc, -1), vf).permute(0, 2, 1, 3).reshape(M, 4096)
    assert _rel(r.attn[:M], o_ref) < 1e-2
    assert _rel(r.o[:M], lin_q(r.attn[:M].float().cpu(), a.o_proj)) < 1e-2
    res1 = res0 + r.o[:M].float().cpu()
    assert torch.equal(r.res[:M].cpu(), res1)
    h2 = norm(res1, layer.post_attention_layernorm.weight)
    gu_ref = torch.cat([lin_q(h2, m.gate_proj), lin_q(h2, m.up_proj)], 1)
    assert _rel(r.gu[:M], gu_ref) < 1e-2
    g, u = r.gu[:M].float().cpu()[:, :4096], r.gu[:M].float().cpu()[:, 4096:]
    assert _rel(r.down[:M], lin_q(g * torch.sigmoid(g) * u, m.down_proj)) < 1e-2


def test_prefill_logits_follow_a_torch_forward(small_models, cuda_device):
    """Whole-model check of the prefill logits.  The random-init network
    amplifies the rare fp8 code differences between the engine and the
    reference quantizer layer after layer, so the bound is loose (cosine
    > 0.99); the per-stage test above carries the tight checks."""
    from ecf8_amd.llm import Qwen3Runner

    cfg, plain, _ = small_models
    B, T = 2, 16
    prompt = _prompt(cfg, B, T)
    r = Qwen3Runner(plain, B, T, T + 1, cuda_device)
    got = r.prefill(prompt).float().cpu()
    ref = _torch_forward(plain, prompt)
    cos = torch.nn.functional.cosine_similarity(got.reshape(-1), ref.reshape(-1), dim=0).item()
    _say(f"[llm] prefill logits cosine {cos:.6f}")
    assert cos > 0.99, cos


@pytest.mark.parametrize("G", [4, 8])
def test_fused_attention_equals_the_unfused_pair(cuda_device, G):
    """decode_attention_fused = qk_norm_rope (T = 1) + decode_attention, bit
    for bit: outputs and the new token's cache rows, at positions inside,
    at the start and at the end of a 256-position split; repeated calls
    and graph replays with a moving position."""
    from ecf8_amd.llm_kernels import (attention_work, decode_attention, decode_attention_fused,
                                      qk_norm_rope)

    dev = cuda_device
    gen = torch.Generator().manual_seed(40 + G)
    B, Hkv, Lmax = 3, 2, 600
    Hq = G * Hkv
    qkv = torch.randn(B, (Hq + 2 * Hkv) * 128, generator=gen).to(torch.bfloat16).to(dev)
    qn = (1 + 0.1 * torch.randn(128, generator=gen)).to(torch.bfloat16).to(dev)
    kn = (1 + 0.1 * torch.randn(128, generator=gen)).to(torch.bfloat16).to(dev)
    cos, sin = (t.to(dev) for t in _rope_tables(Lmax))
    kc0 = (torch.randn(B, Hkv, Lmax, 128, generator=gen) * 2).to(torch.bfloat16).to(dev)
    vc0 = torch.randn(B, Hkv, Lmax, 128, generator=gen).to(torch.bfloat16).to(dev)
    for p0 in (0, 255, 256, 517, Lmax - 1):
        _say(f"[llm] fused attention G={G} pos={p0}")
        pos = torch.tensor([p0], dtype=torch.int32, device=dev)
        # unfused
        kc, vc = kc0.clone(), vc0.clone()
        q = torch.empty(B * Hq * 128, dtype=torch.bfloat16, device=dev)
        qk_norm_rope(qkv, B, 1, Hq, Hkv, qn, kn, 1e-6, cos, sin, pos, q, kc, vc)
        work = attention_work(B, Hq, Lmax, dev)
        oq = torch.empty(pad16(B), Hq * 128, dtype=FP8, device=dev)
        os_ = torch.empty(B, Hq, device=dev)
        ob = torch.empty(B, Hq * 128, dtype=torch.bfloat16, device=dev)
        decode_attention(q, kc, vc, pos, work, oq, os_, Hq, out_bf16=ob)
        # fused, three calls in a row on one work buffer
        kf, vf = kc0.clone(), vc0.clone()
        workf = attention_work(B, Hq, Lmax, dev)
        for _ in range(3):
            oqf = torch.empty_like(oq)
            osf = torch.empty_like(os_)
            obf = torch.empty_like(ob)
            decode_attention_fused(qkv, B, Hq, Hkv, qn, kn, 1e-6, cos, sin, pos, kf, vf, workf,
                                   oqf, osf, out_bf16=obf)
            torch.cuda.synchronize()
            assert torch.equal(kf, kc) and torch.equal(vf, vc)
            assert torch.equal(obf, ob)
            assert torch.equal(osf, os_)
            assert torch.equal(from_tiles(oqf, B, Hq * 128).view(torch.uint8),
                               from_tiles(oq, B, Hq * 128).view(torch.uint8))
    # graph replays with a moving position
    pos = torch.tensor([300], dtype=torch.int32, device=dev)
    kf, vf = kc0.clone(), vc0.clone()
    workf = attention_work(B, Hq, Lmax, dev)
    oqf = torch.empty(pad16(B), Hq * 128, dtype=FP8, device=dev)
    osf = torch.empty(B, Hq, device=dev)
    obf = torch.empty(B, Hq * 128, dtype=torch.bfloat16, device=dev)
    s = torch.cuda.Stream(dev)
    s.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(s):
        decode_attention_fused(qkv, B, Hq, Hkv, qn, kn, 1e-6, cos, sin, pos, kf, vf, workf, oqf,
                               osf, out_bf16=obf)
    torch.cuda.current_stream(dev).wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        decode_attention_fused(qkv, B, Hq, Hkv, qn, kn, 1e-6, cos, sin, pos, kf, vf, workf, oqf,
                               osf, out_bf16=obf)
    for p0 in (301, 302, 511, 512):
        pos.fill_(p0)
        g.replay()
        torch.cuda.synchronize()
        kc, vc = kf.clone(), vf.clone()  # rows below p0 as the replays left them
        q = torch.empty(B * Hq * 128, dtype=torch.bfloat16, device=dev)
        qk_norm_rope(qkv, B, 1, Hq, Hkv, qn, kn, 1e-6, cos, sin, pos, q, kc, vc)
        ob = torch.empty_like(obf)
        decode_attention(q, kc, vc, pos, attention_work(B, Hq, Lmax, dev), torch.empty_like(oqf),
                         torch.empty_like(osf), Hq, out_bf16=ob)
        assert torch.equal(obf, ob), p0


def _skew_exponents(w, frac, exp, seed):
    """e4m3fn weight with ``frac`` of its exponents set to ``exp`` (sign and
    mantissa kept; exponent 15 with mantissa 7 avoided)."""
    b = w.view(torch.uint8).clone()
    rng = np.random.default_rng(seed)
    hit = torch.from_numpy(rng.random(tuple(b.shape)) < frac)
    b[hit] = (b[hit] & 0x87) | (exp << 3)
    return b.view(FP8)


def _spread_exponents(w, seed):
    """e4m3fn weight with exponents drawn uniformly from 1..14 (about 3.8
    bits each under any code), sign and mantissa kept."""
    b = w.view(torch.uint8).clone()
    rng = np.random.default_rng(seed)
    e = torch.from_numpy(rng.integers(1, 15, tuple(b.shape), dtype=np.int64)).to(torch.uint8)
    return ((b & 0x87) | (e << 3)).view(FP8)


def test_retile_keeps_refused_layers_on_decode_then_gemm(cuda_device):
    """Three layers: one the tiled layout holds, one whose LUTs have a
    1-bit code (no automaton table) and one whose down projection needs
    over 3 bits per exponent in its segments.  retile_layers re-tiles the
    first, leaves the other two compressed with their decode hooks, and the
    fused run gives the FP8 model's tokens and logits, eager and
    graph-replayed."""
    from dfloat.run.run import TensorManager
    from ecf8_amd.llm import Qwen3Config, Qwen3Runner, compress_layers, random_model, \
        retile_layers

    cfg = Qwen3Config(**dict(SMALL, layers=3))
    plain, drawn = random_model(cfg, cuda_device, seed=5)
    for name in list(drawn[1]):
        w, s = drawn[1][name]
        drawn[1][name] = (_skew_exponents(w, 0.85, 11, seed=len(name)), s)
    w, s = drawn[2]["mlp.down_proj"]
    drawn[2]["mlp.down_proj"] = (_spread_exponents(w, seed=3), s)
    for i, layer in enumerate(plain.model.layers):
        for name, (w, _s) in drawn[i].items():
            layer.get_submodule(name).weight.data.copy_(w.to(cuda_device))
    comp, _ = random_model(cfg, cuda_device, seed=5)
    compress_layers(comp, drawn)
    retile_layers(comp, drawn)
    untiled = dict(comp._ecf8_untiled)
    assert sorted(untiled) == ["model.layers.1", "model.layers.2"], untiled
    assert "1-bit code" in untiled["model.layers.1"]
    assert "cannot hold a Linear" in untiled["model.layers.2"]
    l0, l1, l2 = comp.model.layers
    assert hasattr(l0, "_ecf8_tiles") and not hasattr(l0, "encoded")
    for lay in (l1, l2):
        assert hasattr(lay, "encoded") and not hasattr(lay, "_ecf8_tiles")
        assert len(lay._forward_pre_hooks) == 1
    B, T, new = 2, 16, 6
    prompt = _prompt(cfg, B, T)
    results = {}
    for name, model in (("fp8", plain), ("fused", comp)):
        for graph in (False, True):
            _say(f"[llm] partial retile {name} graph={graph}")
            TensorManager.clear_device()
            r = Qwen3Runner(model, B, T, T + new, cuda_device)
            if graph:
                r.capture()
            toks = r.generate(prompt, new).cpu()
            results[(name, graph)] = (toks, r.logits.float().cpu())
            del r
    base_t, base_l = results[("fp8", False)]
    for key, (t, l) in results.items():
        assert torch.equal(t, base_t), key
        assert torch.equal(l, base_l), key
