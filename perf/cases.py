"""The work a speech server has this library do, as measurable cases.

The served model pairs a Qwen3-style backbone (hidden 2048, MLP 6144, 16 query and 8 key/value heads of 128,
28 layers) with a 12-layer depth decoder (hidden 1024, MLP 8192, 8 / 2 heads of 128, 16 codebooks of 2051 tokens).
The wider decoder shapes (hidden 2560, MLP 10240, 16 / 4 heads of 256) are the library's other measured geometry.
Per frame a request runs one backbone step and one depth frame; before its first frame it runs the prompt through
the same linears (prefill).  Cases of one layer go through that layer's own entry point; two are whole captured
steps.  All weights are random, with the distributions the benchmark uses.
"""

import math
import os
import sys
import types

import torch
from torch import nn

sys.path.insert(0, os.path.join(os.getcwd(), "breeze-tts-2_amd"))

from breeze_amd import attention as attn  # noqa: E402
from breeze_amd.fp8_linear import Fp8Linear, quantize_module_fp8  # noqa: E402
from breeze_amd.fused.depth_graph import DepthDecodeGraph  # noqa: E402
from breeze_amd.fused.graph import BackboneDecodeGraph  # noqa: E402
from breeze_amd.fused.install import install_fused_backbone, install_fused_depth  # noqa: E402
from breeze_amd.fused.kernels import FusedWeight, rms_gemv  # noqa: E402
from breeze_amd.gemv import EPI_RESIDUAL, EPI_SILU_GATE  # noqa: E402
from breeze_amd.heads import Fp32Linear  # noqa: E402
from breeze_amd.int4_linear import Int4Linear, quantize_module_int4  # noqa: E402
from breeze_amd.sampling import SampleState, sample_cfg  # noqa: E402

DEV = "cuda"
EPS = 1e-6
GROUP = 128
BF16 = torch.bfloat16


def listed():
    return [
        # one projection of one request without guidance: the smallest call there is
        {"name": "linear_int4_m1", "kind": "linear", "fmt": "int4", "M": 1, "N": 2048, "K": 2048},
        # a decoder layer's MLP for a request with classifier-free guidance (conditional + unconditional row)
        {"name": "mlp_int4_m2", "kind": "mlp", "fmt": "int4", "M": 2, "H": 2560, "I": 10240},
        # the same for four such requests in one batch, fp8 weights
        {"name": "mlp_fp8_m8", "kind": "mlp", "fmt": "fp8", "M": 8, "H": 2560, "I": 10240},
        # verification of drafted tokens: a long-row projection over a small batch
        {"name": "linear_int4_m16", "kind": "linear", "fmt": "int4", "M": 16, "N": 2560, "K": 10240},
        # a larger, odd batch of rows
        {"name": "linear_fp8_m27", "kind": "linear", "fmt": "fp8", "M": 27, "N": 10240, "K": 2560},
        # the prompt of one request: a few hundred positions, an odd number of them
        {"name": "prefill_int4_m203", "kind": "linear", "fmt": "int4", "M": 203, "N": 10240, "K": 2560},
        # a long prompt (reference audio and text) over the backbone's MLP
        {"name": "prefill_fp8_m1024", "kind": "linear", "fmt": "fp8", "M": 1024, "N": 6144, "K": 2048},
        # the longest prompt the 2048-position cache takes, with guidance off
        {"name": "prefill_int4_m2048", "kind": "linear", "fmt": "int4", "M": 2048, "N": 2560, "K": 10240},
        # attention of one decode step near the end of a 2048-position cache
        {"name": "attention_s2048", "kind": "attention", "B": 2, "S": 2048, "pos": 1901, "HQ": 16, "HKV": 4, "D": 256},
        # the end of a backbone step: fp32 head, guidance, top-k / top-p sampling of the frame's first token
        {"name": "head_sample_b2", "kind": "head", "B": 2, "K": 2048, "V": 2052, "top_k": 50, "top_p": 0.95},
        # one captured backbone step: 28 layers, int4 MLP, bf16 attention projections, head and guidance
        {"name": "backbone_step", "kind": "backbone", "B": 2, "S": 1024, "pos": 611, "layers": 28, "attn_bits": 16},
        # one captured depth frame: 16 positions through 12 fp8 layers, 15 codebook heads and greedy picks
        {"name": "depth_frame", "kind": "depth", "B": 2, "C": 16, "layers": 12},
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# (out, in) of the projections of the model's layers and of the wider geometry
_SHAPES = [(2048, 2048), (4096, 2048), (6144, 2048), (2048, 6144), (8192, 1024), (1024, 8192), (1024, 1024),
           (4096, 2560), (6144, 2560), (2560, 4096), (10240, 2560), (2560, 10240)]


def draw(rng):
    kind = rng.choice(["linear", "linear", "prefill", "prefill", "mlp", "attention", "head", "backbone", "depth"])
    fmt = rng.choice(["int4", "fp8"])
    if kind in ("linear", "prefill"):
        if rng.random() < 0.3:  # sizes of no particular model
            n, k = 16 * _spread(rng, 16, 640), 128 * _spread(rng, 4, 80)
        else:
            n, k = rng.choice(_SHAPES)
        m = _spread(rng, 1, 32) if kind == "linear" else _spread(rng, 33, 2048)
        return {"kind": "linear", "fmt": fmt, "M": m, "N": n, "K": k}
    if kind == "mlp":
        h, i = rng.choice([(2560, 10240), (2048, 6144), (1024, 8192)])
        return {"kind": "mlp", "fmt": fmt, "M": _spread(rng, 1, 16), "H": h, "I": i}
    if kind == "attention":
        s = rng.choice([17, 512, 1024, 2048])
        hq, hkv, d = rng.choice([(16, 4, 256), (16, 8, 128), (8, 2, 128)])
        return {"kind": "attention", "B": rng.choice([1, 2, 4, 8]), "S": s, "pos": _spread(rng, 1, s - 1),
                "HQ": hq, "HKV": hkv, "D": d}
    if kind == "head":
        return {"kind": "head", "B": rng.choice([1, 2, 4, 8, 16]), "K": rng.choice([1024, 2048, 2560]),
                "V": rng.choice([2051, 2052]), "top_k": _spread(rng, 5, 1000), "top_p": round(rng.uniform(0.8, 1.0), 3)}
    if kind == "backbone":
        s = rng.choice([512, 1024, 2048])
        return {"kind": "backbone", "B": rng.choice([1, 2, 4]), "S": s, "pos": _spread(rng, 16, s - 1),
                "layers": rng.randint(2, 12), "attn_bits": rng.choice([8, 16])}
    return {"kind": "depth", "B": rng.choice([1, 2, 4]), "C": rng.randint(4, 16), "layers": rng.randint(2, 12)}


# ---- what a program has in hand before the call ----------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, device=DEV, generator=g)


def _weight(g, n, k):
    return (_randn(g, n, k) * 0.02).to(BF16)


def _gamma(g, k):
    return (1 + 0.1 * _randn(g, k)).to(BF16)


def _linear(w):
    lin = nn.Linear(w.shape[1], w.shape[0], bias=False, device="meta")
    lin.weight = nn.Parameter(w, requires_grad=False)
    return lin


def _linear_data(case, seed):
    g = _gen(seed)
    return _weight(g, case["N"], case["K"]), _randn(g, case["M"], case["K"]).to(BF16)


def _mlp_data(case, seed):
    g = _gen(seed)
    h, i = case["H"], case["I"]
    x = _randn(g, case["M"], h).to(BF16)
    return _weight(g, i, h), _weight(g, i, h), _weight(g, h, i), _gamma(g, h), x


def _attention_data(case, seed):
    """qkv of the new token, rotary tables, a cache filled up to the position, per-head norm weights."""
    g = _gen(seed)
    b, s, hq, hkv, d = (case[k] for k in ("B", "S", "HQ", "HKV", "D"))
    pos = case["pos"]
    inv = 1.0 / (1e6 ** (torch.arange(0, d, 2, device=DEV, dtype=torch.float64) / d))
    ang = (pos * inv).repeat(2).expand(b, 1, d)
    keys, values = (_randn(g, b, hkv, s, d).to(BF16) for _ in range(2))
    keys[:, :, pos:], values[:, :, pos:] = 0, 0
    at = torch.arange(s, device=DEV)
    pad = torch.randint(0, max(1, min(pos, 8)), (b, 1), device=DEV, generator=g)  # left padding of the batch
    mask = torch.where((at[None] >= pad) & (at[None] <= pos), 0.0, torch.finfo(BF16).min).to(BF16).view(b, 1, 1, s)
    return {"qkv": _randn(g, b, (hq + 2 * hkv) * d).to(BF16), "cos": ang.cos().to(BF16), "sin": ang.sin().to(BF16),
            "pos": torch.tensor([pos], device=DEV), "keys": keys, "values": values, "mask": mask,
            "qn": _gamma(g, d), "kn": _gamma(g, d)}


def _head_data(case, seed):
    g = _gen(seed)
    b, k, v = case["B"], case["K"], case["V"]
    half = max(1, b // 2)
    return {"w": _weight(g, v, k) * 3, "x": _randn(g, b, k).to(BF16),
            "temperature": torch.full((half,), 0.9, device=DEV), "guidance": torch.full((half,), 1.5, device=DEV),
            "top_k": torch.full((half,), case["top_k"], device=DEV, dtype=torch.int64),
            "top_p": torch.full((half,), case["top_p"], device=DEV),
            "do_sample": torch.ones(half, device=DEV, dtype=torch.int64)}


def _stack(g, layers, hidden, inter, hq, hkv, d, positions):
    from transformers import Qwen3Config
    from transformers.models.qwen3.modeling_qwen3 import Qwen3Model

    cfg = Qwen3Config(hidden_size=hidden, intermediate_size=inter, num_attention_heads=hq, num_key_value_heads=hkv,
                      head_dim=d, num_hidden_layers=layers, rms_norm_eps=EPS, max_position_embeddings=positions,
                      vocab_size=64)
    cfg._attn_implementation = "eager"
    with torch.device(DEV):
        model = Qwen3Model(cfg).to(BF16).eval()
    with torch.no_grad():
        for p in model.parameters():
            p.copy_(_gamma(g, p.numel()) if p.dim() == 1 else _weight(g, *p.shape))
            p.requires_grad_(False)
    return model, cfg


def _prepare_backbone(case, seed):
    g = _gen(seed)
    b, s, pos = case["B"], case["S"], case["pos"]
    model, cfg = _stack(g, case["layers"], 2048, 6144, 16, 8, 128, s)
    quantize_module_int4(model)
    install_fused_backbone(types.SimpleNamespace(backbone_model=model), batch_size=b, max_seq_len=s,
                           attn_bits=case["attn_bits"])
    graph = BackboneDecodeGraph(model, _linear(_weight(g, 2052, 2048)), batch_size=b, max_seq_len=s, guidance_scale=1.5)
    x = _randn(g, b, 1, 2048).to(BF16)
    graph.set_step(x, pos)
    graph.capture(num_warmup=1)
    with torch.inference_mode():
        for layer in graph.static_cache.layers:  # the positions before this one
            for t in (layer.keys, layer.values):
                t.copy_(_randn(g, *t.shape))
                t[:, :, pos:] = 0
    return {"kind": "backbone", "graph": graph, "x": x, "pos": pos}


def _prepare_depth(case, seed):
    g = _gen(seed)
    b, c, vocab, width = case["B"], case["C"], 2051, 2048
    model, cfg = _stack(g, case["layers"], 1024, 8192, 8, 2, 128, 64)
    cfg.num_codebooks, cfg.backbone_hidden_size, cfg.vocab_size = c, width, vocab
    model.embed_tokens = nn.Embedding.from_pretrained(_weight(g, c * vocab, width) * 50)
    model.inputs_embeds_projector = _linear(_weight(g, 1024, width))
    model.backbone_hidden_state_projector = None
    # tokens differ in frequency, so logits have a heavy tail, as a trained head's
    head = _randn(g, c - 1, 1024, vocab) * 0.02 * torch.exp(0.7 * _randn(g, c - 1, 1, vocab))
    quantize_module_fp8(model)
    install_fused_depth(types.SimpleNamespace(depth_decoder=types.SimpleNamespace(model=model)), batch_size=b,
                        attn_bits=8)
    decoder = types.SimpleNamespace(model=model, codebooks_head=types.SimpleNamespace(weight=head, num_codebooks=c))
    graph = DepthDecodeGraph(decoder, batch_size=b, do_sample=False, guidance_scale=1.5, debug=True, seed=seed)
    graph.capture(num_warmup=1)
    first = torch.randint(0, vocab, (max(1, b // 2),), device=DEV, generator=g)
    return {"kind": "depth", "graph": graph, "hidden": _randn(g, b, width).to(BF16),
            "first": first if b == 1 else first.repeat(2)}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        w, x = _linear_data(case, seed)
        return {"kind": kind, "mod": (Int4Linear if case["fmt"] == "int4" else Fp8Linear)(_linear(w)), "x": x}
    if kind == "mlp":
        gate, up, down, gamma, x = _mlp_data(case, seed)
        mod, adopt = (Int4Linear, FusedWeight.from_int4) if case["fmt"] == "int4" else (Fp8Linear, FusedWeight.from_fp8)
        mods = [mod(_linear(w)) for w in (gate, up, down)]
        return {"kind": kind, "gu": adopt(*mods[:2], paired=True), "down": adopt(mods[2]), "gamma": gamma, "x": x}
    if kind == "attention":
        return {"kind": kind, **_attention_data(case, seed)}
    if kind == "head":
        d = _head_data(case, seed)
        half = max(1, case["B"] // 2)
        return {"kind": kind, **d, "head": Fp32Linear(_linear(d["w"])), "draws": SampleState(half, DEV, seed),
                "tokens": torch.zeros(case["B"], device=DEV, dtype=torch.int64),
                "cfg": torch.zeros(half, case["V"], device=DEV), "probs": torch.zeros(half, case["V"], device=DEV)}
    return _prepare_backbone(case, seed) if kind == "backbone" else _prepare_depth(case, seed)


# ---- one pass -----------------------------------------------------------------------------------------


@torch.inference_mode()
def run(state):
    s = state
    kind = s["kind"]
    if kind == "linear":
        return s["mod"](s["x"])
    if kind == "mlp":
        mid = rms_gemv(s["x"], s["gu"], s["gamma"], EPS, epilogue=EPI_SILU_GATE)
        return rms_gemv(mid, s["down"], None, epilogue=EPI_RESIDUAL, residual=s["x"])
    if kind == "attention":
        out = attn.attention_step(s["qkv"], s["cos"], s["sin"], s["pos"], s["keys"], s["values"], s["mask"], s["qn"],
                                  s["kn"], EPS)
        return {"out": out, "keys": s["keys"], "values": s["values"]}
    if kind == "head":
        logits = s["head"](s["x"])
        sample_cfg(logits, s["tokens"], s["draws"], temperature=s["temperature"], top_k=s["top_k"], top_p=s["top_p"],
                   do_sample=s["do_sample"], guidance=s["guidance"] if logits.shape[0] > 1 else None, codec_size=2048,
                   cfg_out=s["cfg"], probs_out=s["probs"])
        return {"logits": logits, "cfg": s["cfg"][:, :2048], "probs": s["probs"], "tokens": s["tokens"]}
    g = s["graph"]
    if kind == "backbone":
        out = g.step(s["x"], s["pos"])
        cache = g.static_cache.layers
        return {"cfg_logits": out, "logits": g.logits_buf, "hidden": g.hidden_buf,
                "keys": [layer.keys[:, :, s["pos"]] for layer in cache[:12]],
                "values": [layer.values[:, :, s["pos"]] for layer in cache[:12]]}
    tokens = g.run(s["hidden"], s["first"])
    return {"tokens": tokens, "logits": g.debug_logits}


# ---- what a pass cannot do without --------------------------------------------------------------------


def _wbytes(fmt, n, k):
    """A quantized weight with its scales: 4 bits and a bf16 pair per group of 128, or 8 bits and an fp32 per row;
    or plain bf16."""
    return {"int4": n * k // 2 + 4 * n * (k // GROUP), "fp8": n * k + 4 * n, "bf16": 2 * n * k}[fmt]


def _attention_work(b, n, hq, hkv, d):
    """One token against n attended positions: qkv in, cache rows of the positions read, the new one written, out."""
    nbytes = 2 * b * ((hq + 2 * hkv) * d + 2 * hkv * n * d + 2 * hkv * d + n + hq * d) + 4 * d * b + 4 * d
    return nbytes, 4 * b * hq * n * d


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["M"], case["N"], case["K"]
        return {"bytes": _wbytes(case["fmt"], n, k) + 2 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "mlp":
        m, h, i = case["M"], case["H"], case["I"]
        return {"bytes": _wbytes(case["fmt"], 2 * i, h) + _wbytes(case["fmt"], h, i) + 2 * h + 4 * m * h,
                "flops": 6 * m * h * i}
    if kind == "attention":
        nbytes, flops = _attention_work(case["B"], case["pos"] + 1, case["HQ"], case["HKV"], case["D"])
        return {"bytes": nbytes, "flops": flops}
    if kind == "head":
        b, k, v = case["B"], case["K"], case["V"]
        half = max(1, b // 2)
        return {"bytes": 4 * v * k + 2 * b * k + 4 * b * v + 8 * half * v, "flops": 2 * b * k * v}
    if kind == "backbone":
        b, layers, n = case["B"], case["layers"], case["pos"] + 1
        attn_fmt = "bf16" if case["attn_bits"] == 16 else "fp8"
        a_bytes, a_flops = _attention_work(b, n, 16, 8, 128)
        weights = (_wbytes(attn_fmt, 4096, 2048) + _wbytes(attn_fmt, 2048, 2048) + _wbytes("int4", 12288, 2048)
                   + _wbytes("int4", 2048, 6144))
        params = 2048 * (4096 + 2048 + 3 * 6144)
        return {"bytes": layers * (weights + a_bytes) + 4 * 2052 * 2048 + b * (4 * 2048 + 6 * 2052),
                "flops": layers * (2 * b * params + a_flops) + 2 * b * 2052 * 2048}
    b, layers, c = case["B"], case["layers"], case["C"]
    # the frame's two first positions share one pass over the weights, as a causal start may
    weights = _wbytes("fp8", 1536 + 1024 + 2 * 8192, 1024) + _wbytes("fp8", 1024, 8192)
    steps, positions = c - 1, c
    params = 1024 * (1536 + 1024 + 3 * 8192)
    return {"bytes": steps * (layers * weights + 2 * 2048 * 1024 + 4 * 2051 * 1024) + 2 * positions * b * 2048,
            "flops": 2 * b * (positions * (layers * params + 2048 * 1024) + steps * 1024 * 2051)}


def tolerance(case):
    """About four times what a run differs from the 64-bit result, or, for the captured steps, from a run whose
    inputs moved by one bf16 step in a quarter of their values (no change of any token in eight such frames)."""
    kind = case["kind"]
    if kind == "linear":
        # bf16 results of 32-bit sums 1.7e-3; 2.4e-3 where the effective weight is rounded to bf16 too (prefill)
        return {"rel": 9e-3, "max": 8e-2}
    if kind == "mlp":
        # two such products with a bf16 activation between them: 2.8e-3
        return {"rel": 1.1e-2, "max": 6e-2}
    if kind == "attention":
        # bf16 out of 32-bit softmax sums: 1.7e-3
        return {"rel": 7e-3, "max": 5e-2}
    if kind == "head":
        # 32-bit sums: 1e-7; the probabilities 9e-7, 3e-5 at most
        return {"rel": 1e-5, "max": 2e-4}
    if kind == "backbone":
        # 2.7e-2, 0.15 at most, after 28 layers of bf16 activations
        return {"rel": 1.1e-1, "max": 6e-1}
    # 2.0e-2, 0.41 at most (the heaviest logits), after up to 16 x 12 layers
    return {"rel": 8e-2, "max": 9e-1}


# ---- the same in 64 bits --------------------------------------------------------------------------------


def _int4_weight(w):
    """w_eff in float64 of group-128 min/max int4 with bf16 (scale, zero) pairs."""
    n, k = w.shape
    g = w.float().reshape(n, k // GROUP, GROUP)
    lo, hi = g.amin(-1, keepdim=True), g.amax(-1, keepdim=True)
    s = ((hi - lo) / torch.full_like(hi, 15)).clamp_min(1e-8)  # a division, not a product with 1/15
    q = ((g - lo) / s).round().clamp(0, 15)
    z = lo + 8 * s
    return ((q.double() - 8) * s.to(BF16).double() + z.to(BF16).double()).reshape(n, k)


def _fp8_weight(w):
    s = w.float().abs().amax(1, keepdim=True).clamp_min(1e-12)
    s = s / torch.full_like(s, 448)
    codes = (w.float() / s).clamp(-448, 448).to(torch.float8_e4m3fn)
    return codes.double() * s.double()


def _eff(fmt, w):
    return _int4_weight(w) if fmt == "int4" else _fp8_weight(w)


def _rms(x, gamma):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gamma.double()


def _exact_attention(case, seed):
    d = _attention_data(case, seed)
    b, hq, hkv, dim, pos = (case[k] for k in ("B", "HQ", "HKV", "D", "pos"))
    rows = d["qkv"].double().view(b, hq + 2 * hkv, dim)
    q, k, v = rows[:, :hq], rows[:, hq:hq + hkv], rows[:, hq + hkv:]
    cos, sin = d["cos"].double(), d["sin"].double()

    def rope(t):
        return t * cos + torch.cat([-t[..., dim // 2:], t[..., :dim // 2]], -1) * sin

    q, k = rope(_rms(q, d["qn"])), rope(_rms(k, d["kn"]))
    keys, values = d["keys"].double(), d["values"].double()
    keys[:, :, pos], values[:, :, pos] = k, v
    n = pos + 1
    group = hq // hkv
    kk = keys[:, :, :n].to(BF16).double()  # the cache holds bf16
    scores = torch.matmul(q.view(b, hkv, group, dim), kk.transpose(2, 3).contiguous()) * dim ** -0.5
    p = torch.softmax(scores + d["mask"].double()[..., :n], -1)
    out = torch.matmul(p, values[:, :, :n].contiguous())
    return {"out": out.reshape(b, hq * dim), "keys": keys, "values": values}


def _exact_head(case, seed):
    d = _head_data(case, seed)
    logits = d["x"].double() @ d["w"].double().t().contiguous()
    half = max(1, case["B"] // 2)
    cfg = logits if case["B"] == 1 else logits[half:] + 1.5 * (logits[:half] - logits[half:])
    cfg = cfg[:, :2048].contiguous()
    top, at = torch.topk(cfg / d["temperature"].double().view(-1, 1), case["top_k"])
    p = torch.softmax(top, -1)
    before = torch.cumsum(p, -1) - p
    p = torch.where(before <= d["top_p"].double().view(-1, 1), p, torch.zeros_like(p))
    probs = torch.zeros(half, case["V"], device=DEV, dtype=torch.float64).scatter_(1, at, p / p.sum(-1, keepdim=True))
    return {"logits": logits, "cfg": cfg, "probs": probs, "tokens": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        w, x = _linear_data(case, seed)
        return x.double() @ _eff(case["fmt"], w).t().contiguous()
    if kind == "mlp":
        gate, up, down, gamma, x = _mlp_data(case, seed)
        u = _rms(x.double(), gamma)
        g, v = (u @ _eff(case["fmt"], w).t().contiguous() for w in (gate, up))
        return x.double() + (torch.nn.functional.silu(g) * v) @ _eff(case["fmt"], down).t().contiguous()
    if kind == "attention":
        return _exact_attention(case, seed)
    if kind == "head":
        return _exact_head(case, seed)
    return None  # dozens of layers of 16-bit activations; tokens feed back into what follows
