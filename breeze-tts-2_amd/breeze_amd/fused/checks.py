"""What a decode graph checks before one of its launches stands in for a module."""

from __future__ import annotations

import torch

__all__ = ["is_rmsnorm", "plain_call"]


def plain_call(mod) -> bool:
    """Whether calling the module runs its class's forward and nothing else: no
    forward hook, on it or on every module, and no forward of its own (as
    tools that wrap a module in place leave it)."""
    every = torch.nn.modules.module
    return not (mod._forward_hooks or mod._forward_pre_hooks or every._global_forward_hooks
                or every._global_forward_pre_hooks or "forward" in vars(mod))


@torch.no_grad()
def is_rmsnorm(norm, weight: torch.Tensor, eps: float) -> bool:
    """Whether norm(x), x bf16 [rows, 1, K], is x * rsqrt(mean(x^2) + eps) *
    weight for rows that tell it from its relatives: a mean that is not zero
    (a norm that subtracts it), a scale that differs along the row (one that
    works in groups), and squares as small as eps (another eps, or none)."""
    K = weight.numel()
    g = torch.Generator().manual_seed(0)
    rows = torch.randn(4, K, generator=g)
    rows[0] += 0.5
    rows[1] = torch.linspace(0.01, 3.0, K)
    rows[2] *= torch.linspace(0.1, 4.0, K)
    rows[3] *= max(eps, 1e-12) ** 0.5
    x = rows.to(torch.bfloat16).to(weight.device).unsqueeze(1)
    got = norm(x)
    if not isinstance(got, torch.Tensor) or got.shape != x.shape:
        return False
    f = x.double()
    want = f * torch.rsqrt(f.square().mean(-1, keepdim=True) + eps) * weight.double()
    # two roundings to bf16 (of the normed row, then of its product with the
    # weight) are 2^-8 of the value; the fp32 sums are far below
    return bool(((got.double() - want).abs() <= 2.0 ** -7 * want.abs()).all())
