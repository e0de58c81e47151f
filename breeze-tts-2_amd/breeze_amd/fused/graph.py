"""HIP-graph decode step over a fused backbone (mirrors the decode step of
models/cudagraph/backbone_graph.py:56-320).

One captured graph runs a whole single-token step for a batch of rows:
rotary embedding of the step's position ids, every decoder layer (the fused
layers of install_fused_backbone: GEMVs and the attention step on
libbzgemv.so), the final norm, the fp32 head (Fp32Linear, heads.py) and the
classifier-free-guidance combination of cond / uncond rows.  All inputs live
in static buffers that the host updates in place before each replay:

    inputs_buf      [B, 1, H]   the step's input embeddings
    cache_position  [1]         KV cache slot (shared by the rows)
    position_ids    [B, 1]      per-row RoPE positions
    attn_mask       [B, 1, 1, S] additive, rebuilt on the device from
                                 pad_lens and the position
                                 (backbone_graph.py:240-252)

Around the layers lie two launches: the mask and the rotary tables
(bz_step_tables), and the final norm, the head and the guidance combination
(bz_norm_head_f32).  Both stand in only for modules that compute just that,
which is checked against the modules at set-up and before a capture; others,
and modules with forward hooks, run as they are.

The layers are called directly (not through the model's forward), so no
mask construction or shape logic of the model runs inside the capture.
"""

from __future__ import annotations

import torch
from torch import nn

from ..heads import NORM_HEAD_MAX_K, NORM_HEAD_MAX_ROWS, Fp32Linear, norm_head_f32
from .checks import is_rmsnorm, plain_call
from .install import static_cache, zero_cache
from .kernels import step_tables

__all__ = ["BackboneDecodeGraph"]


class BackboneDecodeGraph:
    def __init__(self, backbone_model: nn.Module, lm_head: nn.Module, *, batch_size: int = 2,
                 max_seq_len: int = 1024, guidance_scale: float = 1.0):
        self.model = backbone_model
        self.lm_head = Fp32Linear(lm_head) if isinstance(lm_head, nn.Linear) else lm_head
        self.batch_size = batch_size
        self.half = batch_size // 2 if batch_size >= 2 else batch_size
        self.max_seq_len = max_seq_len
        self.guidance_scale = float(guidance_scale)
        p = next(backbone_model.parameters())
        dev, dtype = p.device, p.dtype
        self.device = dev
        cfg = backbone_model.config
        self.static_cache = static_cache(cfg, max_seq_len, batch_size)
        self.cache_position = torch.zeros(1, dtype=torch.long, device=dev)
        self.position_ids = torch.zeros(batch_size, 1, dtype=torch.long, device=dev)
        self.pad_lens = torch.zeros(batch_size, dtype=torch.long, device=dev)
        self.kv_indices = torch.arange(max_seq_len, device=dev)
        self.mask_min = torch.finfo(dtype).min
        self.attn_mask = torch.full((batch_size, 1, 1, max_seq_len), self.mask_min, dtype=dtype, device=dev)
        self.inputs_buf = torch.zeros(batch_size, 1, cfg.hidden_size, dtype=dtype, device=dev)
        self.hidden_buf = torch.zeros(batch_size, 1, cfg.hidden_size, dtype=dtype, device=dev)
        vocab = self.lm_head.out_features
        self.logits_buf = torch.zeros(batch_size, vocab, dtype=torch.float32, device=dev)
        self.cfg_logits_buf = torch.zeros(self.half, vocab, dtype=torch.float32, device=dev)
        self._rotary_class = self._norm_class = self._tables = None
        self._find_stand_ins()
        self.graph = None

    # -- what the two launches around the layers may stand in for -------------------
    #
    # That a class of modules computes what its launch does is found by running
    # it (at set-up and before every capture); everything the launch reads of
    # the module is read when the step runs.

    def _rotary(self):
        """(inv_freq, scaling) of a rotary embedding of the default type, else None."""
        rot = self.model.rotary_emb
        inv, scale = getattr(rot, "inv_freq", None), getattr(rot, "attention_scaling", 1.0)
        if (self.device.type != "cuda" or self.inputs_buf.dtype not in (torch.bfloat16, torch.float32)
                or not plain_call(rot) or getattr(rot, "rope_type", None) != "default"
                or not isinstance(inv, torch.Tensor) or not inv.is_floating_point() or inv.dim() != 1
                or inv.device != self.device):
            return None
        inv = inv.detach()  # the module widens it to fp32 on every call, and so does the kernel
        if inv.dtype not in (torch.float32, torch.bfloat16):
            inv = inv.float()
        return inv.contiguous(), float(scale)

    def _norm(self):
        """(weight, eps) of a norm with an RMSNorm's parameters that
        bz_norm_head_f32 can run with this head, else None."""
        norm, head, H = self.model.norm, self.lm_head, self.inputs_buf.shape[-1]
        w, eps = getattr(norm, "weight", None), getattr(norm, "variance_epsilon", None)
        if (self.device.type != "cuda" or type(head) is not Fp32Linear or w is None or eps is None
                or not plain_call(norm) or not plain_call(head) or self.inputs_buf.dtype != torch.bfloat16
                or w.dtype != torch.bfloat16 or w.shape != (H,) or not w.is_contiguous() or w.device != self.device
                or head.in_features != H or H > NORM_HEAD_MAX_K or self.batch_size > NORM_HEAD_MAX_ROWS
                or (self.batch_size > 1 and self.batch_size % 2)):
            return None
        return w.detach(), float(eps)

    def _find_stand_ins(self) -> None:
        """Which classes of rotary embedding and norm the launches stand in for:
        one whose tables have the same bits at a spread of positions, and one
        that is an RMSNorm."""
        self._rotary_class = self._norm_class = None
        facts = self._rotary()
        if facts is not None:
            B, D, dt = self.batch_size, 2 * facts[0].numel(), self.inputs_buf.dtype
            if self._tables is None or self._tables[0].shape[-1] != D:
                self._tables = [torch.zeros(B, 1, D, dtype=dt, device=self.device) for _ in range(2)]
            mask, same = torch.empty_like(self.attn_mask), True
            with torch.no_grad():
                for p in (0, 1, self.max_seq_len // 3, self.max_seq_len - 1):
                    ids = torch.full((B, 1), p, dtype=torch.long, device=self.device)
                    step_tables(torch.zeros_like(ids[:, 0]), ids[:1, 0], self.mask_min, mask, ids, *facts, *self._tables)
                    want = self.model.rotary_emb(self.inputs_buf, ids)
                    same = same and all(w.dtype == dt and w.shape == t.shape and torch.equal(w, t)
                                        for w, t in zip(want, self._tables))
            if same:
                self._rotary_class = type(self.model.rotary_emb)
        facts = self._norm()
        if facts is not None and is_rmsnorm(self.model.norm, *facts):
            self._norm_class = type(self.model.norm)

    # -- device-side state ---------------------------------------------------------

    def _set_attention_mask(self) -> None:
        """valid[b, s] = pad_lens[b] <= s <= position (in place, no host sync)."""
        kv = self.kv_indices
        valid = (kv >= self.pad_lens.unsqueeze(1)) & (kv <= self.cache_position)
        self.attn_mask.fill_(self.mask_min)
        self.attn_mask[:, 0, 0, :].masked_fill_(valid, 0.0)

    def _decode_step(self) -> None:
        h = self.inputs_buf
        ints = (self.pad_lens, self.cache_position, self.position_ids)
        rotary = self._rotary() if type(self.model.rotary_emb) is self._rotary_class else None
        if rotary is not None and 2 * rotary[0].numel() == self._tables[0].shape[-1] \
                and all(t.dtype == torch.long and t.is_contiguous() for t in ints):
            pe = self._tables
            step_tables(self.pad_lens, self.cache_position, self.mask_min, self.attn_mask, self.position_ids, *rotary,
                        *pe)
        else:
            self._set_attention_mask()
            pe = self.model.rotary_emb(h, self.position_ids)
        for layer in self.model.layers:
            h = layer(h, attention_mask=self.attn_mask, position_ids=self.position_ids,
                      past_key_values=self.static_cache, use_cache=True, cache_position=self.cache_position,
                      position_embeddings=pe)
            h = h[0] if isinstance(h, tuple) else h
        norm = self._norm() if type(self.model.norm) is self._norm_class else None
        if norm is not None and h.dtype == torch.bfloat16 and isinstance(self.guidance_scale, (int, float)):
            norm_head_f32(h[:, -1, :], *norm, self.lm_head.weight, out=self.logits_buf,
                          normed=self.hidden_buf[:, -1, :], cfg=self.cfg_logits_buf, guidance=self.guidance_scale)
            return
        h = self.model.norm(h)
        self.hidden_buf.copy_(h)
        self.logits_buf.copy_(self.lm_head(self.hidden_buf[:, -1, :].float()))
        if self.batch_size >= 2:
            cond, uncond = self.logits_buf[: self.half], self.logits_buf[self.half: 2 * self.half]
            self.cfg_logits_buf.copy_(uncond + self.guidance_scale * (cond - uncond))
        else:
            self.cfg_logits_buf.copy_(self.logits_buf[: self.half])

    # -- host API -----------------------------------------------------------------

    def set_step(self, inputs_embeds: torch.Tensor, position: int, position_ids=None) -> None:
        """Stage one step's inputs: embeddings [B, 1, H], cache slot `position`
        and per-row RoPE positions (default: `position` for every row)."""
        self.inputs_buf.copy_(inputs_embeds)
        self.cache_position.fill_(position)
        if position_ids is None:
            self.position_ids.fill_(position)
        else:
            self.position_ids.copy_(torch.as_tensor(position_ids).reshape(self.batch_size, 1))

    @torch.inference_mode()
    def capture(self, num_warmup: int = 2) -> None:
        """Warm up (loads the library, sizes the allocator) and capture one step
        on a side stream, as backbone_graph.py:287-320.  The warm-up writes into
        the cache at the staged position; reset() clears it."""
        self._find_stand_ins()
        self._captured = (self._rotary(), self._norm())  # replays read these, replaced in their modules or not
        for _ in range(num_warmup):
            self._decode_step()
        torch.cuda.synchronize(self.device)
        self.graph = torch.cuda.CUDAGraph()
        s = torch.cuda.Stream(device=self.device)
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            with torch.cuda.graph(self.graph, stream=s):
                self._decode_step()
        torch.cuda.current_stream().wait_stream(s)
        torch.cuda.synchronize(self.device)

    @torch.inference_mode()
    def reset(self) -> None:
        zero_cache(self.static_cache)

    @torch.inference_mode()
    def step(self, inputs_embeds: torch.Tensor, position: int, position_ids=None) -> torch.Tensor:
        """One decode step (graph replay once captured); returns the CFG logits
        buffer [B / 2, vocab] fp32 (valid until the next step)."""
        self.set_step(inputs_embeds, position, position_ids)
        if self.graph is None:
            self._decode_step()
        else:
            self.graph.replay()
        return self.cfg_logits_buf
