"""DiT blocks on the CPU: what the HIP kernels do not take (here: CPU
tensors) runs in torch, forward, backward and forward-mode."""

from __future__ import annotations

import pytest
import torch

from ecf8_amd.dit import DoubleBlock, FluxConfig, SingleBlock, _Lin, FluxDiT


def _block(cls, cfg):
    torch.manual_seed(3)
    blk = cls(cfg)
    for mod in blk.modules():
        if isinstance(mod, _Lin):  # bf16 weights as a fused decode leaves them
            mod.__dict__["_w_bf16"] = (torch.randn(mod.out_features, mod.in_features) * 0.02).bfloat16()
    return blk


@pytest.mark.parametrize("cls", [DoubleBlock, SingleBlock])
def test_blocks_run_and_differentiate_in_torch(cls):
    cfg = FluxConfig(hidden=64, heads=2, head_dim=32, mlp=128, axes=(8, 12, 12))
    blk = _block(cls, cfg)
    cos, sin = FluxDiT.rope_tables(type("D", (), {"cfg": cfg})(), 3, 2, 3, "cpu")
    img, txt, emb = (torch.randn(2, n, 64).bfloat16() for n in (6, 3, 1))
    emb = emb[:, 0]
    args = (img, txt, emb) if cls is DoubleBlock else (torch.cat([txt, img], 1), emb)
    leaf = args[0].clone().requires_grad_()
    out = blk(leaf, *args[1:], cos, sin)
    first = out[0] if isinstance(out, tuple) else out
    first.float().sum().backward()
    assert first.shape == args[0].shape and bool(torch.isfinite(leaf.grad).all())
    with torch.no_grad():
        again = blk(*args, cos, sin)
    assert torch.equal(again[0] if isinstance(again, tuple) else again, first)


def test_kernels_refuse_what_they_do_not_take():
    from ecf8_amd import dit_kernels as DK

    x, v = torch.randn(1, 4, 64).bfloat16(), torch.randn(1, 64).bfloat16()
    assert DK.modulate(x, v, v) is None and DK.gated_add(x, v, x) is None
    assert not DK._takes((x,))
    with torch.autocast("cpu"):
        assert DK._untracked()  # only CUDA autocast changes what the CUDA path computes
    assert DK._untracked()
    with torch.autograd.forward_ad.dual_level():
        assert not DK._untracked()
    seen = []

    def f(t):
        seen.append(DK._takes((t,)))
        return t

    torch.vmap(f)(x)
    assert seen == [False]


def test_own_forwards_and_function_modes_are_kept():
    """A Linear whose forward was replaced on the instance runs that forward;
    a function mode keeps calls in torch, a default device alone does not."""
    from torch.overrides import TorchFunctionMode

    from ecf8_amd import guards
    from ecf8_amd.dit import _AdaNorm

    class Watch(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    norm = _AdaNorm(8, 2)
    norm.linear = torch.nn.Linear(8, 16).bfloat16()
    assert guards.bare(norm.linear, torch.nn.Linear)
    norm.linear.forward = lambda x: torch.full((x.shape[0], 16), 3.0)
    assert all(bool((t == 3.0).all()) for t in norm(torch.randn(2, 8).bfloat16()))
    with Watch():
        assert not guards.untracked()
    with torch.device("cpu"):
        assert guards.untracked()
