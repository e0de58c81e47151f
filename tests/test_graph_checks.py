"""The checks behind the decode graphs' stand-in launches (CPU)."""

from __future__ import annotations

import pytest
import torch
from torch import nn

from breeze_amd.fused.checks import is_rmsnorm, plain_call


class _Norm(nn.Module):
    """RMSNorm in the model's roundings, or a relative of it."""

    def __init__(self, K, kind, eps=1e-6):
        super().__init__()
        self.kind, self.variance_epsilon = kind, eps
        g = torch.Generator().manual_seed(K)
        self.weight = nn.Parameter((1 + 0.1 * torch.randn(K, generator=g)).to(torch.bfloat16), requires_grad=False)

    def forward(self, x):
        f = x.float()
        if self.kind == "mean":
            f = f - f.mean(-1, keepdim=True)
        eps = {"other_eps": 4 * self.variance_epsilon, "no_eps": 0.0}.get(self.kind, self.variance_epsilon)
        if self.kind == "groups":
            v = f.unflatten(-1, (4, -1))
            f = (v * torch.rsqrt(v.square().mean(-1, keepdim=True) + eps)).flatten(-2)
        else:
            f = f * torch.rsqrt(f.square().mean(-1, keepdim=True) + eps)
        w = self.weight + 1 if self.kind == "offset" else self.weight
        out = w * f.to(x.dtype) if self.kind != "one_rounding" else (w.float() * f).to(x.dtype)
        return out[0] if self.kind == "shape" else out


@pytest.mark.parametrize("K", [64, 512, 1024, 2048, 2560, 4096])
@pytest.mark.parametrize("kind,plain", [("rms", True), ("one_rounding", True), ("mean", False), ("groups", False),
                                        ("offset", False), ("other_eps", False), ("no_eps", False), ("shape", False)])
def test_is_rmsnorm(K, kind, plain):
    for eps in (1e-6, 1e-5):
        norm = _Norm(K, kind, eps)
        assert is_rmsnorm(norm, norm.weight, eps) is plain


def test_is_rmsnorm_of_the_model():
    from transformers.models.qwen3.modeling_qwen3 import Qwen3RMSNorm

    norm = Qwen3RMSNorm(2048, 1e-6).to(torch.bfloat16)
    assert is_rmsnorm(norm, norm.weight, norm.variance_epsilon)


def test_plain_call():
    mod = nn.Embedding(4, 4)
    assert plain_call(mod)
    for register in (mod.register_forward_hook, mod.register_forward_pre_hook,
                     nn.modules.module.register_module_forward_hook, nn.modules.module.register_module_forward_pre_hook):
        handle = register(lambda *a: None)
        assert not plain_call(mod)
        handle.remove()
        assert plain_call(mod)
    mod.forward = lambda ids: None
    assert not plain_call(mod)
