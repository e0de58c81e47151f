"""fp32 heads through the C ABI against the oracle (float64), on the GPU.
Bar: 1e-5 of the largest output (fp32 products and sums over K <= 2560)."""

from __future__ import annotations

import numpy as np
import pytest
import torch
from torch import nn

from oracle import bz_oracle as O
from tests._util import f32

from breeze_amd import heads as Hd

pytestmark = pytest.mark.gpu

TOL = 1e-5
DEV = "cuda"


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 9])
@pytest.mark.parametrize("K,N", [(1024, 2051), (2048, 2052), (2560, 8192), (64, 7)])
def test_head_f32_matches_oracle(M, K, N):
    rng = np.random.default_rng(M * 31 + K)
    x = rng.standard_normal((M, K)).astype(np.float32)
    w = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    got = f32(Hd.head_f32(torch.from_numpy(x).to(DEV), torch.from_numpy(w).to(DEV)))
    assert O.rel_err(got, O.linear_f32_ref(x, w)) <= TOL


def test_head_f32_device_index_selects_matrix_and_out_of_range_is_zero():
    rng = np.random.default_rng(3)
    C, N, K = 5, 300, 256
    w = rng.standard_normal((C, N, K)).astype(np.float32)
    x = rng.standard_normal((2, K)).astype(np.float32)
    wd, xd = torch.from_numpy(w).to(DEV), torch.from_numpy(x).to(DEV)
    for pos in (1, 3, 5):
        idx = torch.tensor([pos], device=DEV)
        got = f32(Hd.head_f32(xd, wd, index=idx, index_offset=-1))
        assert O.rel_err(got, O.linear_f32_ref(x, w[pos - 1])) <= TOL
    for pos in (0, 6, -3):
        got = f32(Hd.head_f32(xd, wd, index=torch.tensor([pos], device=DEV), index_offset=-1))
        assert not got.any()


def test_fp32_linear_matches_torch_fp32():
    torch.manual_seed(0)
    lin = nn.Linear(2048, 2052, bias=False)
    head = Hd.Fp32Linear(lin)
    x = torch.randn(2, 1, 2048).to(torch.bfloat16)
    got = head(x.to(DEV))
    assert got.dtype == torch.float32 and got.shape == (2, 1, 2052)
    ref = O.linear_f32_ref(x.float().reshape(2, 2048).numpy(), lin.weight.detach().numpy())
    assert O.rel_err(f32(got).reshape(2, 2052), ref) <= TOL


class _CodebooksHead(nn.Module):
    """Same parameters as models/breeze.py:590-596 (weight [C - 1, hidden, vocab])."""

    def __init__(self, hidden, num_codebooks, vocab):
        super().__init__()
        self.num_codebooks = num_codebooks
        self.weight = nn.Parameter(torch.randn(num_codebooks - 1, hidden, vocab) * 0.02)


@pytest.mark.parametrize("with_position", [False, True])
def test_fp32_codebooks_head(with_position):
    torch.manual_seed(1)
    ref_head = _CodebooksHead(1024, 16, 2051)
    head = Hd.Fp32CodebooksHead(ref_head)
    B, L = 2, (1 if with_position else 15)
    hidden = torch.randn(B, L, 1024).to(torch.bfloat16)
    cp = torch.tensor([7]) if with_position else None
    got = head(hidden.to(DEV), None if cp is None else cp.to(DEV))
    ref = O.codebooks_head_ref(hidden.float().numpy(), ref_head.weight.detach().numpy(),
                               None if cp is None else cp.numpy())
    assert got.shape == (B, L, 2051)
    assert O.rel_err(f32(got), ref) <= TOL


def test_codebooks_head_graph_replays_follow_device_position():
    """Captured once; the cache position changes between replays (as in the
    depth decoder's graph) and every replay uses its codebook."""
    torch.manual_seed(2)
    ref_head = _CodebooksHead(1024, 16, 2051)
    head = Hd.Fp32CodebooksHead(ref_head)
    hidden = torch.randn(2, 1, 1024, device=DEV)
    cp = torch.ones(1, dtype=torch.int64, device=DEV)
    out = torch.empty(2, 1, 2051, device=DEV)
    head(hidden, cp)
    torch.cuda.synchronize()
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(st):
        with torch.cuda.graph(g, stream=st):
            out.copy_(head(hidden, cp))
    torch.cuda.current_stream().wait_stream(st)
    torch.cuda.synchronize()
    w = ref_head.weight.detach().numpy()
    for p in (1, 15, 4, 9):
        cp.fill_(p)
        g.replay()
        torch.cuda.synchronize()
        ref = O.codebooks_head_ref(f32(hidden), w, np.array([p]))
        assert O.rel_err(f32(out), ref) <= TOL, p


def test_install_fp32_heads():
    class _Model(nn.Module):
        def __init__(self):
            super().__init__()
            self.lm_head = nn.Linear(256, 2052, bias=False)
            self.depth_decoder = nn.Module()
            self.depth_decoder.codebooks_head = _CodebooksHead(128, 4, 2051)

    m = _Model()
    assert Hd.install_fp32_heads(m) == 2
    assert isinstance(m.lm_head, Hd.Fp32Linear)
    assert isinstance(m.depth_decoder.codebooks_head, Hd.Fp32CodebooksHead)
    assert Hd.install_fp32_heads(m) == 0


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N,K", [(1, 4), (9, 252), (2051, 1024), (64, 1028), (2052, 2048), (17, 2052), (33, 2560), (33, 2564), (40, 4096)])
def test_norm_head_equals_its_parts(M, N, K):
    """norm_head_f32 against bz_rmsnorm, head_f32 and the guidance formula: the
    same bits for the first two (edges of its 256-k pieces and of its two
    instances), one rounding of the combination apart for the last."""
    from breeze_amd.gemv import rmsnorm
    from breeze_amd.heads import head_f32, norm_head_f32

    g = torch.Generator(device="cuda").manual_seed(N + K + M)
    x = torch.randn(M, K + 3, device="cuda", generator=g).to(torch.bfloat16)[:, 3:]
    gamma = (1 + 0.1 * torch.randn(K, device="cuda", generator=g)).to(torch.bfloat16)
    w = torch.randn(3, N, K, device="cuda", generator=g)
    index = torch.tensor([2], device="cuda")
    normed = torch.zeros(M, K, device="cuda", dtype=torch.bfloat16)
    out = torch.zeros(M, N, device="cuda")
    cfg = torch.zeros(max(1, M // 2), N, device="cuda") if M != 3 else None
    norm_head_f32(x, gamma, 1e-6, w, out=out, index=index, index_offset=-1, normed=normed, cfg=cfg, guidance=1.5)
    xn = rmsnorm(x, gamma, 1e-6)
    want = head_f32(xn, w, index=index, index_offset=-1)
    assert torch.equal(normed, xn)
    assert torch.equal(out, want)
    assert torch.equal(head_f32(x, w, index=index, index_offset=-1),  # bf16 rows, widened by the kernel
                       head_f32(x.float().clone(memory_format=torch.contiguous_format), w, index=index, index_offset=-1))
    if cfg is not None:
        h = max(1, M // 2)
        ref = want if M == 1 else want[h:].double() + 1.5 * (want[:h].double() - want[h:].double())
        mag = want.abs().max()
        assert bool(((cfg.double() - ref).abs() <= 2.0 ** -22 * 4 * mag).all())
