"""Graph and compile integration on the GPU.

* BackboneDecodeGraph (the reference's BackboneGraph decode step,
  models/cudagraph/backbone_graph.py:254-320) over a fused 3-layer Qwen3
  backbone with an fp32 head and CFG, captured once and replayed over
  positions with per-row padding, against the CPU float32 model running the
  same layers eagerly (bar 1e-2 on the CFG logits).
* torch.compile(fullgraph=True) over a module holding Int4Linear / Fp8Linear
  (the reference compiles its depth-decoder layers,
  models/cudagraph/depth_decoder_graph.py:164-192): the GEMV custom op traces
  without graph breaks and gives the eager result."""

from __future__ import annotations

import copy
import types

import numpy as np
import pytest
import torch
from torch import nn

from oracle import bz_oracle as O

from breeze_amd import fp8_linear as F8
from breeze_amd import int4_linear as I4
from breeze_amd.fused.graph import BackboneDecodeGraph
from breeze_amd.fused.install import install_fused_backbone, static_cache

pytestmark = pytest.mark.gpu

TOL = 1e-2


def _model(layers=3, seed=7):
    from transformers import Qwen3Config
    from transformers.models.qwen3.modeling_qwen3 import Qwen3Model

    cfg = Qwen3Config(hidden_size=512, intermediate_size=1024, num_attention_heads=8, num_key_value_heads=2,
                      head_dim=128, num_hidden_layers=layers, rms_norm_eps=1e-6, max_position_embeddings=4096,
                      vocab_size=64)
    cfg._attn_implementation = "eager"
    torch.manual_seed(seed)
    m = Qwen3Model(cfg).float().eval()
    with torch.no_grad():
        for p in m.parameters():
            (p.normal_(0, 0.03) if p.dim() == 2 else p.normal_(1, 0.1))
            p.copy_(p.to(torch.bfloat16).float())
    head = nn.Linear(512, 130, bias=False)
    with torch.no_grad():
        head.weight.normal_(0, 0.05)
    return cfg, m, head


def test_backbone_decode_graph_matches_cpu_model():
    cfg, ref, head = _model()
    gpu = copy.deepcopy(ref).to("cuda", torch.bfloat16)
    install_fused_backbone(types.SimpleNamespace(backbone_model=gpu), batch_size=2, max_seq_len=48)
    B, S, scale = 2, 48, 1.7
    g = BackboneDecodeGraph(gpu, copy.deepcopy(head).cuda(), batch_size=B, max_seq_len=S, guidance_scale=scale)
    g.pad_lens.copy_(torch.tensor([0, 2]))
    gen = torch.Generator().manual_seed(3)
    xs = [torch.randn(B, 1, 512, generator=gen).to(torch.bfloat16).float() for _ in range(10)]
    g.set_step(xs[0].cuda(), 0)
    g.capture(num_warmup=1)
    g.reset()

    c_ref = static_cache(cfg, S, B)
    mask = torch.full((B, 1, 1, S), torch.finfo(torch.float32).min)
    for t, x in enumerate(xs):
        out = g.step(x.to("cuda", torch.bfloat16), t).float().cpu().numpy()
        pid = torch.full((B, 1), t)
        kv = torch.arange(S)
        valid = (kv >= torch.tensor([0, 2]).unsqueeze(1)) & (kv <= t)
        mask.fill_(torch.finfo(torch.float32).min)
        mask[:, 0, 0, :] = mask[:, 0, 0, :].masked_fill(valid, 0.0)
        with torch.no_grad():
            h = x
            pe = ref.rotary_emb(h, pid)
            for layer in ref.layers:
                h = layer(h, attention_mask=mask, position_ids=pid, past_key_values=c_ref, use_cache=True,
                          position_embeddings=pe)
                h = h[0] if isinstance(h, tuple) else h
            h = ref.norm(h)[:, -1, :]
        logits = O.linear_f32_ref(h.numpy(), head.weight.detach().numpy())
        cfg_ref = logits[1:2] + scale * (logits[0:1] - logits[1:2])
        if t >= 2:  # row 1 attends to nothing before position 2
            assert O.rel_err(out, cfg_ref) <= TOL, t


def test_compile_fullgraph_with_quantized_linears():
    torch.manual_seed(0)

    class _MLP(nn.Module):
        def __init__(self):
            super().__init__()
            self.gate_proj = nn.Linear(512, 1024, bias=False)
            self.up_proj = nn.Linear(512, 1024, bias=False)
            self.down_proj = nn.Linear(1024, 512, bias=False)

        def forward(self, x):
            return self.down_proj(torch.nn.functional.silu(self.gate_proj(x)) * self.up_proj(x))

    for quant in (I4.quantize_module_int4, F8.quantize_module_fp8):
        m = _MLP().to("cuda", torch.bfloat16)
        quant(m, min_bytes=0)
        x = torch.randn(2, 1, 512, device="cuda").to(torch.bfloat16)
        eager = m(x)
        compiled = torch.compile(m, fullgraph=True, backend="aot_eager")
        got = compiled(x)
        assert torch.equal(got, eager)
        np.testing.assert_array_equal(compiled(x * 2).float().cpu().numpy(), m(x * 2).float().cpu().numpy())


@pytest.mark.parametrize("quant", ["int4", "fp8"])
def test_inductor_compile_then_graph_capture(quant):
    """The reference's depth-decoder flow (models/cudagraph/
    depth_decoder_graph.py:164-192; test_fp8_linear.py:38-63): a module
    holding Int4Linear / Fp8Linear compiled with the default backend
    (inductor, mode="default", fullgraph=True), then captured in a HIP graph
    and replayed.  The GEMV custom op stays one opaque launch; inductor
    generates the glue (SiLU-mul, residual add) itself, in fp32 where eager
    torch rounds the SiLU to bf16 first, so the compiled module is held to
    the 1e-2 bar against the uncompiled one, and every graph replay to the
    compiled module's eager result bit for bit."""
    torch.manual_seed(1)

    class _Block(nn.Module):
        def __init__(self):
            super().__init__()
            self.gate_proj = nn.Linear(512, 1024, bias=False)
            self.up_proj = nn.Linear(512, 1024, bias=False)
            self.down_proj = nn.Linear(1024, 512, bias=False)

        def forward(self, x):
            return x + self.down_proj(torch.nn.functional.silu(self.gate_proj(x)) * self.up_proj(x))

    m = _Block().to("cuda", torch.bfloat16)
    (I4.quantize_module_int4 if quant == "int4" else F8.quantize_module_fp8)(m, min_bytes=0)
    x = torch.randn(2, 1, 512, device="cuda").to(torch.bfloat16)
    eager = m(x)
    compiled = torch.compile(m, mode="default", fullgraph=True)
    want = compiled(x)
    assert O.rel_err(want.float().cpu().numpy(), eager.float().cpu().numpy()) <= TOL
    static_x = x.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):  # warm-up calls outside the capture
            compiled(static_x)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        out = compiled(static_x)
    torch.cuda.synchronize()
    for rep in range(3):
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), rep
        _ = (x.float() * 3).sum().item()  # eager work between the replays
    static_x.copy_(x * 2)
    g.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, compiled(x * 2))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,S,D", [(1, 1, 2), (2, 257, 128), (3, 1024, 256), (2, 300, 514)])
def test_step_tables(B, S, D, dt):
    """The mask exactly; cos and sin of the same fp32 angle within one rounding
    of the output type and 4 ulp of the fp32 functions."""
    from breeze_amd.fused.kernels import step_tables

    dev, low = "cuda", torch.finfo(dt).min
    pad = torch.tensor([0, 3, S][:B], device=dev)
    pos = torch.tensor([min(200, S - 1)], device=dev)
    ids = torch.tensor([[7], [0], [40000]][:B], device=dev)
    inv = 1.0 / 1e6 ** (torch.arange(0, D, 2, device=dev).float() / D)
    mask = torch.full((B, 1, 1, S), 5.0, device=dev, dtype=dt)
    cos, sin = (torch.full((B, 1, D), 5.0, device=dev, dtype=dt) for _ in range(2))
    step_tables(pad, pos, low, mask, ids, inv, 1.5, cos, sin)
    rounded = inv.to(torch.bfloat16)  # frequencies as a model cast to bf16 holds them
    same = [torch.zeros_like(t) for t in (mask, cos, sin, cos, sin)]
    step_tables(pad, pos, low, same[0], ids, rounded, 1.5, *same[1:3])
    step_tables(pad, pos, low, same[0], ids, rounded.float(), 1.5, *same[3:])
    assert torch.equal(same[1], same[3]) and torch.equal(same[2], same[4])
    s = torch.arange(S, device=dev)
    valid = (s >= pad.view(B, 1)) & (s <= pos)
    assert torch.equal(mask.view(B, S), torch.where(valid, 0.0, low).to(dt))
    a = (ids.view(B, 1).float() * inv).double().repeat(1, 2)
    tol = 1.5 * (2.0 ** -8 if dt == torch.bfloat16 else 0.0) + 1.5 * 2.0 ** -21
    for t, f in ((cos, torch.cos), (sin, torch.sin)):
        assert float((t.view(B, D).double() - 1.5 * f(a)).abs().max()) <= tol


class _MeanNorm(nn.Module):
    """A norm with RMSNorm's attributes that subtracts the mean (as transformers' CohereLayerNorm)."""

    def __init__(self, weight, eps):
        super().__init__()
        self.weight, self.variance_epsilon = weight, eps

    def forward(self, x):
        f = x.float()
        f = f - f.mean(-1, keepdim=True)
        f = f * torch.rsqrt(f.square().mean(-1, keepdim=True) + self.variance_epsilon)
        return (self.weight.float() * f).to(x.dtype)


def _mean_norm(m):
    m.norm = _MeanNorm(m.norm.weight, m.norm.variance_epsilon)


def _linear_rope(m):
    """Positions divided by 3: not the default rotary type."""
    m.rotary_emb.rope_type = "linear"
    m.rotary_emb.inv_freq = m.rotary_emb.inv_freq / 3


def _graph(B, change=None, scale=1.7, S=48):
    cfg, ref, head = _model()
    if change is not None:
        change(ref)
    gpu = copy.deepcopy(ref).to("cuda", torch.bfloat16)
    # (a module's own cast would round the frequencies)
    gpu.rotary_emb.inv_freq = ref.rotary_emb.inv_freq.float().cuda()
    install_fused_backbone(types.SimpleNamespace(backbone_model=gpu), batch_size=B, max_seq_len=S)
    g = BackboneDecodeGraph(gpu, copy.deepcopy(head).cuda(), batch_size=B, max_seq_len=S, guidance_scale=scale)
    return cfg, ref, head, g


def _inputs(B, n, seed=3):
    gen = torch.Generator().manual_seed(seed)
    return [torch.randn(B, 1, 512, generator=gen).to(torch.bfloat16).float() for _ in range(n)]


@pytest.mark.parametrize("B,change", [(1, None), (4, None), (6, None), (2, _mean_norm), (2, _linear_rope), (6, _linear_rope)],
                         ids=["1", "4", "6", "mean", "rope", "rope6"])
def test_backbone_stand_ins_and_fallbacks_match_cpu_model(B, change):
    """The launches around the layers and what takes their place: more rows
    than the fused head takes, a norm that is no RMSNorm, other rotary tables.
    CFG logits against the CPU float32 model."""
    S, scale = 48, 1.7
    cfg, ref, head, g = _graph(B, change, scale, S)
    pads = torch.arange(B) % 3
    g.pad_lens.copy_(pads)
    xs = _inputs(B, 8)
    g.set_step(xs[0].cuda(), 0)
    g.capture(num_warmup=1)
    g.reset()
    c_ref = static_cache(cfg, S, B)
    kv, half = torch.arange(S), max(1, B // 2)
    for t, x in enumerate(xs):
        out = g.step(x.to("cuda", torch.bfloat16), t).float().cpu().numpy()
        pid = torch.full((B, 1), t)
        valid = (kv >= pads.unsqueeze(1)) & (kv <= t)
        mask = torch.where(valid, 0.0, torch.finfo(torch.float32).min).view(B, 1, 1, S)
        with torch.no_grad():
            h, pe = x, ref.rotary_emb(x, pid)
            for layer in ref.layers:
                h = layer(h, attention_mask=mask, position_ids=pid, past_key_values=c_ref, use_cache=True,
                          position_embeddings=pe)
                h = h[0] if isinstance(h, tuple) else h
            h = ref.norm(h)[:, -1, :]
        logits = O.linear_f32_ref(h.numpy(), head.weight.detach().numpy())
        want = logits if B == 1 else logits[half:] + scale * (logits[:half] - logits[half:])
        if t >= 2:  # a padded row attends to nothing before position 2
            assert O.rel_err(out, want) <= TOL, t


@pytest.mark.parametrize("what", ["norm", "rotary_emb", "lm_head"])
def test_backbone_step_runs_forward_hooks(what):
    """A module with a forward hook is called, and what the hook returns counts."""
    _, _, _, g = _graph(2)
    x = _inputs(2, 1)[0].to("cuda", torch.bfloat16)
    g.step(x, 5)
    plain = (g.hidden_buf.clone(), g.logits_buf.clone())
    mod, seen = g.lm_head if what == "lm_head" else getattr(g.model, what), []

    def hook(m, args, out):
        seen.append(tuple(t * 0.5 for t in out) if isinstance(out, tuple) else out * 0.5)
        return seen[-1]

    handle = mod.register_forward_hook(hook)
    g.step(x, 5)
    assert len(seen) == 1
    if what == "norm":
        assert torch.equal(g.hidden_buf, seen[0])
    elif what == "lm_head":
        assert torch.equal(g.logits_buf, seen[0])
    else:
        assert not torch.equal(g.logits_buf, plain[1])
    handle.remove()
    g.step(x, 5)
    assert torch.equal(g.hidden_buf, plain[0]) and torch.equal(g.logits_buf, plain[1])


def _new_inv_freq(m):
    m.rotary_emb.inv_freq = m.rotary_emb.inv_freq * 0.5


def _new_scaling(m):
    m.rotary_emb.attention_scaling = 0.75


def _new_eps(m):
    m.norm.variance_epsilon = 0.5


def _new_norm(m):
    m.norm = _MeanNorm(m.norm.weight, 1e-6)


def _fp32_norm(m):
    m.norm.weight = nn.Parameter(m.norm.weight.detach().float() * 1.5, requires_grad=False)


@pytest.mark.parametrize("captured", [False, True])
@pytest.mark.parametrize("change", [_new_inv_freq, _new_scaling, _new_eps, _new_norm, _fp32_norm])
def test_backbone_step_follows_its_modules(change, captured):
    """A module changed after the graph was built counts in the next eager
    step and in the next capture, as in a graph built after the change."""
    x = _inputs(2, 1)[0].to("cuda", torch.bfloat16)
    got = []
    for late in (True, False):
        _, _, _, g = _graph(2, None)
        if not late:  # the same change before the graph is built
            change(g.model)
            g = BackboneDecodeGraph(g.model, g.lm_head, batch_size=2, max_seq_len=48, guidance_scale=1.7)
        else:
            change(g.model)
        g.set_step(x, 5)
        if captured:
            g.capture(num_warmup=1)
            g.reset()
        got.append((g.step(x, 5).clone(), g.hidden_buf.clone()))
    assert torch.isfinite(got[0][0]).all()
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    _, _, _, g = _graph(2)
    assert not torch.equal(g.step(x, 5), got[0][0])
