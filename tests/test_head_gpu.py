"""GPU checks of the ends of a decode step (include/ecf8_head.h) against
torch: the bf16 linear of a few rows, the greedy token, the embedding."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _rand(shape, seed, dev):
    g = torch.Generator(device=dev).manual_seed(seed)
    return torch.randn(shape, generator=g, device=dev).to(torch.bfloat16)


@pytest.mark.parametrize("M,N,K,bias", [
    (1, 16, 32, False), (2, 48, 64, True), (15, 4096, 1024, True), (16, 4112, 2048, False),
    (7, 128, 4096, True), (16, 5000 * 16, 96, False), (3, 3072, 3072, True), (9, 1040, 1056, False)])
def test_small_linear_matches_fp64(cuda_device, M, N, K, bias):
    """Panels below, at and above one per CU, steps that do not fill the 16
    waves, a strided x; fp32 sums of K products (K 2^-24 of the product of
    norms) and one bf16 rounding (2^-8)."""
    from ecf8_amd.head_kernels import small_linear

    x = _rand((M, K + 8), M + K, cuda_device)[:, :K]
    w = _rand((N, K), N + K, cuda_device)
    b = _rand((N,), N, cuda_device) if bias else None
    got = small_linear(x, w, b).double()
    want = x.double() @ w.double().t() + (b.double() if bias else 0.0)
    norms = x.double().norm(dim=1)[:, None] * w.double().norm(dim=1)[None]
    assert bool(((got - want).abs() <= want.abs() * 2.0 ** -8 * 1.01 + norms * K * 2.0 ** -24).all())


@pytest.mark.parametrize("K", [32, 96, 1056, 2048])
def test_small_linear_keeps_infinities(cuda_device, K):
    """An infinite weight or input in the last step of K: no step past K
    turns it into a NaN."""
    from ecf8_amd.head_kernels import small_linear

    x, w = _rand((3, K), 5, cuda_device), _rand((32, K), 6, cuda_device)
    x[:, -1] = 2.0
    w[7, -1], w[9, -1] = float("inf"), float("-inf")
    got = small_linear(x, w)
    assert bool((got[:, 7] == float("inf")).all()) and bool((got[:, 9] == float("-inf")).all())
    assert not bool(got.isnan().any())


def test_small_linear_leaves_the_rest_to_the_library(cuda_device, monkeypatch):
    """Rows past 16, K or N off its steps, other dtypes, autocast: the
    library's result; autograd through the kernel: the library's gradients."""
    from ecf8_amd import head_kernels as HK

    calls = []
    monkeypatch.setattr(HK, "_launch", lambda *a, _f=HK._launch: (calls.append(1), _f(*a))[1])
    w = _rand((64, 128), 1, cuda_device)
    x = _rand((4, 128), 2, cuda_device)
    for a, b in ((_rand((17, 128), 3, cuda_device), w), (x.t().contiguous().t(), w),
                 (x[:, :120].contiguous(), w[:, :120].contiguous()), (x, w[:60]),
                 (x.float(), w.float()), (x[None], w)):
        assert torch.equal(HK.small_linear(a, b), F.linear(a, b))
    with torch.autocast("cuda", dtype=torch.float16):
        assert HK.small_linear(x, w).dtype == torch.float16
    assert not calls
    bias = _rand((64,), 4, cuda_device)
    grads = []
    for fn in (HK.small_linear, F.linear):
        leaves = [t.clone().requires_grad_() for t in (x, w, bias)]
        fn(*leaves).float().square().sum().backward()
        grads.append([t.grad for t in leaves])
    assert calls
    for a, b in zip(*grads):
        assert float((a.float() - b.float()).norm() / b.float().norm()) <= 2.0 ** -7


@pytest.mark.parametrize("B,V", [(1, 1), (3, 7), (2, 64), (16, 1001), (5, 4096), (33, 151936)])
def test_greedy_emit_matches_argmax(cuda_device, B, V):
    """Many exact ties (logits on a coarse grid), both zeros, infinities and
    NaN; rows aligned and not; the counters move and a full row is kept."""
    from ecf8_amd.head_kernels import greedy_emit, greedy_work

    x = (_rand((B, V), V, cuda_device) * 2).round()
    x[:, ::3] *= -0.0 if V < 64 else 1.0
    if B > 1:
        x[1, V // 2] = float("nan")
        x[0, V - 1] = float("inf")
    tokens = torch.full((B, 3), -1, dtype=torch.int64, device=cuda_device)
    nxt = torch.zeros(B, dtype=torch.int64, device=cuda_device)
    step = torch.ones(1, dtype=torch.int64, device=cuda_device)
    pos = torch.full((1,), 7, dtype=torch.int32, device=cuda_device)
    work = greedy_work(B, cuda_device)
    want = torch.tensor([int((r != r).nonzero()[0]) if bool((r != r).any())
                         else int((r == r.max()).nonzero()[0]) for r in x.cpu().float()])
    for i, advance in enumerate((1, 0, 1)):  # the third call finds the row full
        greedy_emit(x, work, tokens, nxt, step, pos, advance)
        assert torch.equal(nxt.cpu(), want) and int(step) == 2 + i
    assert int(pos) == 9
    assert bool((tokens[:, 0] == -1).all())
    assert torch.equal(tokens[:, 1].cpu(), want) and torch.equal(tokens[:, 2].cpu(), want)


@pytest.mark.parametrize("B,H", [(1, 8), (16, 4096), (3, 2056)])
def test_embed_rows_matches_embedding(cuda_device, B, H):
    from ecf8_amd.head_kernels import embed_rows

    table = _rand((50, H), H, cuda_device)
    tok = torch.randint(0, 50, (B,), device=cuda_device)
    out = torch.full((B + 1, H), 5.0, device=cuda_device)
    embed_rows(tok, table, out)
    assert torch.equal(out[:B], F.embedding(tok, table).float()) and bool((out[B] == 5.0).all())


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("what", ["token", "negative", "step"])
def test_decode_step_refuses_bad_state_at_the_next_call(cuda_device, what, graph):
    """A token outside the vocabulary or a step past the token buffer stays
    inside the kernels' bounds checks and makes the runner's next call raise;
    after that the runner works on."""
    from ecf8_amd._lib import ECF8Error
    from ecf8_amd.llm import Qwen3Config, Qwen3ForCausalLM, Qwen3Runner
    from ecf8_amd.synth import quantize_fp8_blockwise

    cfg = Qwen3Config(layers=1, intermediate=4096, vocab=128)
    model = Qwen3ForCausalLM(cfg).to(cuda_device)
    for name, (o, i, sigma) in cfg.linear_shapes().items():
        lin = model.model.layers[0].get_submodule(name)
        w, s = quantize_fp8_blockwise(sigma * torch.randn(o, i, device=cuda_device))
        lin.weight, lin.weight_scale_inv = torch.nn.Parameter(w, requires_grad=False), s
    with torch.no_grad():
        r = Qwen3Runner(model, 2, 4, 16, cuda_device)
        prompt = torch.randint(0, 128, (2, 4))
        r.prefill(prompt)
        if graph:
            r.capture()
        step = r.graph.replay if graph else r.decode_step
        want = r.generate(prompt, 3).clone()
        if what == "step":
            r.step.fill_(r.tokens.shape[1])
        else:
            r.next_tok[1] = 128 if what == "token" else -1
        tokens = r.tokens.clone()
        step()
        torch.cuda.synchronize()
        if what == "step":
            assert torch.equal(r.tokens, tokens)
        with pytest.raises(ECF8Error, match="vocabulary"):
            r.decode_step()
        for call in (r.capture, lambda: r.prefill(prompt), lambda: r.generate(prompt, 3)):
            r.refused.fill_(1)  # raising cleared it
            with pytest.raises(ECF8Error, match="vocabulary"):
                call()
        assert torch.equal(r.generate(prompt, 3), want)
