"""The prefill GEMM over the tiled formats (bz_gemm_tiled): argument checks on
the CPU, results on the GPU against the float64 product with the oracle's
effective weight, at the edges of its tiles."""

from __future__ import annotations

import itertools

import numpy as np
import pytest
import torch

from oracle import bz_oracle as O
from tests._util import Fp8Case, Int4Case, bf16_tensor, f32

from breeze_amd import _lib
from breeze_amd import gemv as G

FAKE = 1 << 20  # never dereferenced: the calls below fail validation


@pytest.mark.parametrize("kw,status", [
    ({"wfmt": 5}, _lib.ERR_INVALID_ARG), ({"wfmt": 0}, _lib.ERR_INVALID_ARG), ({"M": 0}, _lib.ERR_INVALID_ARG),
    ({"x": None}, _lib.ERR_INVALID_ARG), ({"out_dtype": 2}, _lib.ERR_INVALID_ARG), ({"ldx": 120}, _lib.ERR_INVALID_ARG),
    ({"ldo": 40}, _lib.ERR_INVALID_ARG), ({"cfg": -1}, _lib.ERR_INVALID_ARG), ({"cfg": 3}, _lib.ERR_INVALID_ARG),
    ({"cfg": 8 | 4 << 8}, _lib.ERR_INVALID_ARG), ({"cfg": 2 | 1 << 8 | 2 << 16, "K": 512, "ldx": 512}, _lib.ERR_INVALID_ARG),
    ({"N": 40}, _lib.ERR_SHAPE), ({"K": 192, "ldx": 192}, _lib.ERR_SHAPE), ({"wfmt": 6, "K": 96}, _lib.ERR_SHAPE),
    ({"x": FAKE + 8}, _lib.ERR_ALIGNMENT), ({"ldx": 132}, _lib.ERR_ALIGNMENT), ({"out": FAKE + 1}, _lib.ERR_ALIGNMENT),
    ({"ldx": (1 << 22) + 8}, _lib.ERR_UNSUPPORTED),
])
def test_arguments(kw, status):
    d = dict(wfmt=4, x=FAKE, ldx=128, M=40, w=FAKE, N=48, K=128, out=FAKE, ldo=48, out_dtype=0, ws=None, wsb=0, cfg=0)
    d.update(kw)
    assert _lib.lib().bz_gemm_tiled(d["wfmt"], d["x"], d["ldx"], d["M"], d["w"], d["N"], d["K"], d["out"], d["ldo"],
                                    d["out_dtype"], d["ws"], d["wsb"], d["cfg"], None) == status


def test_workspace_covers_the_slices():
    for wf, m, n, k, s in itertools.product((4, 6), (33, 300), (48, 2560), (128, 2176), (1, 2, 5)):
        got = _lib.lib().bz_gemm_workspace(wf, m, n, k, 2 | 1 << 8 | s << 16)
        steps = -(-k // 256)
        per = -(-steps // min(s, steps))
        slices = -(-steps // per)
        assert got == (slices * m * n * 4 if slices > 1 else 0)
        assert _lib.lib().bz_gemm_workspace(wf, m, n, k, 0) % 4 == 0
    assert _lib.lib().bz_gemm_workspace(5, 33, 48, 128, 0) == 0


def _weight(fmt, n, k):
    w = (np.random.default_rng(n + k).standard_normal((n, k)) * 0.02).astype(np.float32)
    if fmt == "int4":
        c = Int4Case(w, 128)
        return G.pack_tiled(G.W_INT4_ZP, c.d_packed, k, G.W_INT4_TILED, sc0=c.d_sz), G.W_INT4_TILED, c.w_zp
    c = Fp8Case(w)
    return G.pack_tiled(G.W_FP8, c.d_codes, k, G.W_FP8_TILED, sc0=c.d_scale), G.W_FP8_TILED, c.w_eff


def _check(out, x, w_eff, out_rounding=2.0 ** -8):
    """Each result within the rounding of the output, of an int4 weight to
    bf16 (2^-9 of each product) and of K fp32 additions."""
    x, w = x.astype(np.float64), w_eff.astype(np.float64)
    ref, mag = x @ w.T, np.abs(x) @ np.abs(w).T
    bound = out_rounding * np.abs(ref) + (2.0 ** -9 + x.shape[1] * 2.0 ** -23) * mag + 1e-30
    assert np.all(np.abs(f32(out) - ref) <= bound)


def _launch(xt, ldx, m, buf, wf, n, k, dtype, cfg):
    out = torch.full((m, n + 8), float("nan"), device="cuda", dtype=dtype)
    need = _lib.lib().bz_gemm_workspace(wf, m, n, k, cfg)
    ws = torch.full((max(need, 16) // 4,), float("nan"), device="cuda")
    _lib.check(_lib.lib().bz_gemm_tiled(wf, xt.data_ptr(), ldx, m, buf.data_ptr(), n, k, out.data_ptr(), n + 8,
                                        0 if dtype == torch.bfloat16 else 1, ws.data_ptr(), need, cfg,
                                        torch.cuda.current_stream().cuda_stream), "bz_gemm_tiled")
    assert torch.isnan(out[:, n:].float()).all()  # nothing past the row
    return out[:, :n]


# one row block, a partial column tile, several; odd units of K (fp8: also odd tiles)
SHAPES = [("int4", 16, 128), ("int4", 208, 384), ("int4", 400, 2176), ("fp8", 16, 64), ("fp8", 208, 448), ("fp8", 400, 2176)]


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,n,k", SHAPES)
def test_every_tile_shape(fmt, n, k):
    """Rows around each tile's edge, x inside a wider buffer of NaN, every
    tile shape, one and several K slices."""
    buf, wf, w_eff = _weight(fmt, n, k)
    for m, mt in ((33, 2), (65, 4), (95, 6), (97, 6), (129, 8)):
        wide = torch.full((m, k + 64), float("nan"), device="cuda", dtype=torch.bfloat16)
        bits = O.f32_to_bf16_bits(np.random.default_rng(m).standard_normal((m, k)).astype(np.float32))
        wide[:, :k] = bf16_tensor(bits)
        for nt, s in itertools.product((1, 2, 3, 4), (1, 3)):
            if mt * nt > 24:
                continue
            dtype = torch.float32 if nt == 2 else torch.bfloat16
            out = _launch(wide, k + 64, m, buf, wf, n, k, dtype, mt | nt << 8 | s << 16)
            _check(out, O.bf16_bits_to_f32(bits), w_eff, 2.0 ** -8 if dtype == torch.bfloat16 else 0.0)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,m,n,k", [("int4", 33, 1024, 8192), ("fp8", 33, 1024, 8192), ("int4", 203, 2560, 1280),
                                       ("fp8", 700, 1024, 1024), ("int4", 2048, 512, 512)])
def test_rule_layouts_and_replays(fmt, m, n, k):
    """The rule's launch shape through dequant_matmul: rows far apart, columns
    strided, an expanded row, a call that autograd follows, and a captured
    call replayed with eager work between."""
    buf, wf, w_eff = _weight(fmt, n, k)
    bits = O.f32_to_bf16_bits(np.random.default_rng(m).standard_normal((m, k)).astype(np.float32))
    x, xf = bf16_tensor(bits), O.bf16_bits_to_f32(bits)
    want = G.dequant_matmul(x, buf, wf, n, k)
    _check(want, xf, w_eff)
    assert torch.equal(G.dequant_matmul(x.t().contiguous().t(), buf, wf, n, k), want)
    assert torch.equal(G.dequant_matmul(x.repeat(1, 2)[:, :k], buf, wf, n, k), want)
    assert torch.equal(G.dequant_matmul(x[:1].expand(m, k), buf, wf, n, k)[m - 1], want[0])
    xg = x.clone().requires_grad_(True)
    y = G.dequant_matmul(xg, buf, wf, n, k)
    _check(y, xf, w_eff)
    y.float().sum().backward()
    assert xg.grad is not None
    g = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(g, stream=side):
        out = G.dequant_matmul(x, buf, wf, n, k)
    for _ in range(3):
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(G.dequant_matmul(x, buf, wf, n, k), want)
