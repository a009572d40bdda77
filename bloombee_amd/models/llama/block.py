"""Server-side LLaMA decoder block on the gfx950 op library.

Replaces the reference's OptimizedLlamaDecoderLayer + FLEX_LlamaAttention/MLP
stack (models/llama/block.py:149-861, models/llama/flex_llama.py:434-793) with
a flat MI355X-native block:

  * projections via ops.linear (hand-written products for decode and some hundred
    rows, hipBLASLt beyond) with QKV and gate/up fused into single GEMMs (fewer,
    larger GEMMs — xGMI/HBM sizing),
  * hand-written HIP kernels for everything fused: rmsnorm(+residual), RoPE,
    paged KV write, paged decode/prefill attention, SwiGLU,
  * one paged KV pool shared across local layers (kv/paged.py), no
    ValueHolder grids, no per-layer load/store streams: weights are resident
    in 288 GB HBM by default; the offload tier is a separate module.

Two forward paths (by design, mirroring the reference's split between
iterate_rpc_inference and run_rpc_forward/backward):
  forward_inference — HIP kernels + paged KV, no autograd.
  forward_train     — differentiable steps of ops/training.py (fp32 softmax):
                      kernels with their gradients for bf16 on the device, torch
                      operations elsewhere. Used by the fine-tuning RPCs;
                      gradients flow to inputs/prompts only (server weights
                      frozen, ref backend.py:106-109).
"""
from __future__ import annotations

import math
from typing import Optional, Tuple

import torch

from bloombee_amd import ops
from bloombee_amd.kv.paged import SessionHandle, context_bound
from bloombee_amd.models.base import ModelConfig
from bloombee_amd.ops import training


class RopeTables:
    """Shared host-precomputed cos/sin tables, materialized per device."""

    def __init__(self, config: ModelConfig):
        self.config = config
        cos, sin = ops.rope_cos_sin(
            config.head_dim, config.max_position_embeddings,
            theta=config.rope_theta, scaling=config.rope_scaling,
        )
        self._cos, self._sin = cos, sin
        self._cache = {}

    def get(self, device: torch.device):
        key = str(device)
        if key not in self._cache:
            self._cache[key] = (self._cos.to(device), self._sin.to(device))
        return self._cache[key]


class LlamaBlock(torch.nn.Module):
    def __init__(self, config: ModelConfig, layer_index: int = 0,
                 rope: Optional[RopeTables] = None):
        super().__init__()
        self.config = config
        self.layer_index = layer_index
        H = config.hidden_size
        D = config.head_dim
        Hq, Hkv = config.num_attention_heads, config.num_key_value_heads
        I = config.intermediate_size
        dt = config.dtype
        self.Hq, self.Hkv, self.D, self.I = Hq, Hkv, D, I
        self.scale = 1.0 / math.sqrt(D)

        def p(*shape):
            return torch.nn.Parameter(torch.empty(*shape, dtype=dt), requires_grad=False)

        self.input_norm_w = p(H)
        self.qkv_w = p((Hq + 2 * Hkv) * D, H)     # fused q|k|v
        self.o_w = p(H, Hq * D)
        self.post_norm_w = p(H)
        self.gate_up_w = p(2 * I, H)              # fused gate|up
        self.down_w = p(H, I)
        self.rope = rope if rope is not None else RopeTables(config)

    @torch.no_grad()
    def init_random(self, seed: Optional[int] = None):
        """Random-init weights. Generates on the parameters' current device —
        device-side RNG for resident blocks (seconds for 70B-class shards vs
        minutes of host randn + transfer). Same (device kind, seed) => same
        weights, which is what the multi-rank parity argument needs."""
        s = seed if seed is not None else 1234 + self.layer_index
        dev = self.input_norm_w.device
        gen = torch.Generator(device=dev).manual_seed(s)
        std = 0.02 / math.sqrt(2 * self.config.num_hidden_layers)
        for name, w in self.named_parameters():
            if name.endswith("norm_w"):
                w.fill_(1.0)
            else:
                w.copy_(torch.randn(w.shape, generator=gen, dtype=torch.float32,
                                    device=dev).mul_(std).to(w.dtype))
        return self

    def _fuse_norm_gate(self, hidden) -> bool:
        """All four decode GEMMs must be decode-shaped (<= 32 rows, K%256,
        N%64); W4/LoRA blocks keep the separate-norm path, as do blocks whose
        weights are streamed in as they were stored (offload/weights.py): what
        is folded into those is lost with the next binding."""
        return (getattr(self, "_w4", None) is None
                and getattr(self, "lora_delta", None) is None
                and (getattr(self, "_norm_folded", False)
                     or not getattr(self, "streamed", False))
                and ops.fuse_norm_linear_ok(hidden, self.qkv_w)
                and self.I % 256 == 0 and (2 * self.I) % 64 == 0
                and (self.Hq * self.D) % 256 == 0
                and self.config.hidden_size % 64 == 0)

    def _fused_tail(self, hidden, attn) -> torch.Tensor:
        """What follows attention in a decode-shaped step: h2 = hidden + o(attn)
        via the GEMM's residual epilogue; the post-attention rmsnorm and the
        gated product ride gate_up."""
        h2 = ops.linear(attn, self.o_w, residual=hidden)
        m = ops.linear_swiglu(h2, self.gate_up_w, self.config.rms_norm_eps)
        return ops.linear(m, self.down_w, residual=h2)

    def span_norms(self):
        """Norm weights of q and k heads for a span's launch, empty without any; None
        where a block does more than such a launch."""
        if type(self).forward_inference is not _LLAMA_STEP:
            return None
        none = self.qkv_w.new_empty(0)
        return none, none

    @torch.no_grad()
    def fold_norm_weights(self):
        """Reparameterize for the fused-norm decode path: qkv_w <- qkv_w *
        input_norm_w, gate_up_w <- gate_up_w * post_norm_w (f32 product,
        one bf16 round), norm weights <- 1. rms_norm with unit weight is
        mathematically unchanged on EVERY path (train, prefill, CPU), and
        the decode GEMM then only applies the per-row 1/rms in its
        epilogue, from the squares of the rows that it has at hand, instead
        of per-element weight scaling, which cost 4 to 8 us a GEMM."""
        if getattr(self, "_norm_folded", False):
            return
        self._norm_fold_orig = (self.input_norm_w.detach().clone(),
                                self.post_norm_w.detach().clone())
        self.qkv_w.data = (self.qkv_w.float()
                           * self.input_norm_w.float()).to(self.qkv_w.dtype)
        self.gate_up_w.data = (self.gate_up_w.float()
                               * self.post_norm_w.float()).to(self.gate_up_w.dtype)
        self.input_norm_w.data.fill_(1.0)
        self.post_norm_w.data.fill_(1.0)
        self._norm_folded = True

    @torch.no_grad()
    def unfold_norm_weights(self):
        """Best-effort inverse of fold_norm_weights (division re-rounds:
        ~1 ulp drift on the projections). Needed before attaching LoRA
        adapters trained against the original parameterization."""
        if not getattr(self, "_norm_folded", False):
            return
        inw, pnw = self._norm_fold_orig
        self.input_norm_w.data.copy_(inw)
        self.post_norm_w.data.copy_(pnw)
        den_i = inw.float().abs().clamp_min(1e-6) * inw.float().sign().where(
            inw.float() != 0, torch.ones_like(inw.float()))
        den_p = pnw.float().abs().clamp_min(1e-6) * pnw.float().sign().where(
            pnw.float() != 0, torch.ones_like(pnw.float()))
        self.qkv_w.data = (self.qkv_w.float() / den_i).to(self.qkv_w.dtype)
        self.gate_up_w.data = (self.gate_up_w.float() / den_p).to(self.gate_up_w.dtype)
        self._norm_folded = False

    @torch.no_grad()
    def quantize_weights_q4(self, keep_full: bool = False):
        """Pack the four projection weights into 4-bit group codes
        (quant4_pack layout); decode GEMMs then stream ~3.5x fewer bytes
        through w4_gemm.hip (FlexGen-style compression ON the compute
        path — the reference only compresses weights at rest,
        flexgen_utils/compression.py:94-210). keep_full=False drops the
        bf16 weights (4x memory; the block becomes inference-only and
        prefill-shaped GEMMs dequantize on the fly)."""
        self._w4 = {}
        for name in ("qkv_w", "o_w", "gate_up_w", "down_w"):
            w = getattr(self, name).detach()
            packed, scale, zero = ops.quant4_pack(w)
            N = w.shape[0]
            self._w4[name] = (packed.reshape(N, -1).contiguous(),
                              scale.reshape(N, -1).half().contiguous(),
                              zero.reshape(N, -1).half().contiguous(), N)
            if not keep_full:
                getattr(self, name).data = torch.empty(
                    0, dtype=w.dtype, device=w.device)
        return self

    def _lin(self, x, w, name, **kw):
        """ops.linear + optional active-LoRA delta (utils/peft.py).
        Quantized blocks (quantize_weights_q4) route through the 4-bit
        weight-stream kernel instead."""
        w4 = getattr(self, "_w4", None)
        if w4 is not None and name in w4:
            packed, scale, zero, N = w4[name]
            y = ops.linear_w4(x, packed, scale, zero, N, **kw)
        else:
            y = ops.linear(x, w, **kw)
        ld = getattr(self, "lora_delta", None)
        if ld is not None:
            d = ld(name, x)
            if d is not None:
                y = y + d
        return y

    def _plain_weights(self) -> bool:
        """Projections are products with the weights as they are, nothing else."""
        return (getattr(self, "_w4", None) is None
                and getattr(self, "lora_delta", None) is None)

    def _attended(self, attn, hidden):
        """h2 = hidden + o(attn) and its post-attention norm."""
        eps = self.config.rms_norm_eps
        if self._plain_weights():
            return ops.linear_norm(attn, self.o_w, hidden, self.post_norm_w, eps)
        return ops.rms_norm_residual(self._lin(attn, self.o_w, "o_w"), hidden,
                                     self.post_norm_w, eps)

    def _gated(self, y):
        """The gated product of gate_up's result."""
        if self._plain_weights():
            return ops.linear_gated(y, self.gate_up_w)
        return ops.swiglu(self._lin(y, self.gate_up_w, "gate_up_w"))

    # ------------------------------------------------------------------
    # inference path (HIP kernels, paged KV)
    # ------------------------------------------------------------------
    @torch.no_grad()
    def forward_inference(
        self,
        hidden: torch.Tensor,              # (B, T, H) bf16
        kv: SessionHandle,
        start_pos: torch.Tensor,           # (B,) int32 — absolute pos of token 0
        position_ids: Optional[torch.Tensor] = None,  # (B, T) int32
        tree_mask: Optional[torch.Tensor] = None,     # (B, T, T) bool, spec verify
    ) -> torch.Tensor:
        B, T, H = hidden.shape
        Hq, Hkv, D = self.Hq, self.Hkv, self.D
        cfg = self.config

        # Decode-shaped GPU steps fold both per-layer rmsnorms into the
        # decode GEMMs, the rotation with the K/V write into the first one and
        # the gated product into the third: a launch there costs more than
        # most of these steps do. W4/LoRA blocks and prefill keep the separate
        # steps.
        fuse_norm = self._fuse_norm_gate(hidden)
        if fuse_norm and not getattr(self, "_norm_folded", False):
            self.fold_norm_weights()   # one-time reparameterization
        cos, sin = self.rope.get(hidden.device)
        kp = kv.k_pages(self.layer_index)
        vp = kv.v_pages(self.layer_index)
        pt = kv.page_table()
        # mixed-device sessions (host KV prefix + device recent segment,
        # kv.swap_in_as_prefix): paged indices are LOCAL to the device pool
        # but rotary positions must stay ABSOLUTE
        off = getattr(kv, "pos_offset", 0)
        if off and position_ids is None:
            position_ids = (start_pos.view(B, 1) + off
                            + torch.arange(T, device=hidden.device)
                            .view(1, T)).int()
        # fused RoPE + paged KV write on the GEMM output, then attention
        # reads q in place and emits the O-projection input — no transposes
        if fuse_norm:
            qkv = ops.linear_rope_kv(hidden, self.qkv_w, cfg.rms_norm_eps, Hq,
                                     Hkv, cos, sin, position_ids, kp, vp, pt,
                                     start_pos)
        else:
            x = ops.rms_norm(hidden, self.input_norm_w, cfg.rms_norm_eps)
            if self._plain_weights():
                qkv = ops.linear_rope_kv_rows(x, self.qkv_w, Hq, Hkv, cos, sin,
                                              position_ids, kp, vp, pt, start_pos)
            else:
                qkv = self._lin(x, self.qkv_w, "qkv_w")    # (B, T, (Hq+2Hkv)D)
                ops.rope_kv_write_(qkv, Hq, Hkv, cos, sin, position_ids, kp, vp,
                                   pt, start_pos)
        hp = (kv.host_prefix(self.layer_index)
              if hasattr(kv, "host_prefix") else None)
        if hp is not None:
            # exact two-segment merge (ref _mixed_device_attention): the
            # host prefix is attended on the CPU, the recent segment via
            # the paged pool; decode-only (backend gates T == 1)
            D_ = self.D
            q = (qkv[..., : Hq * D_].view(B, T, Hq, D_)
                 .permute(0, 2, 1, 3).contiguous())
            attn = ops.attn_paged_mixed(q, kp, vp, pt, start_pos + T,
                                        hp[0], hp[1], self.scale)
            attn = attn.permute(0, 2, 1, 3).reshape(B, T, Hq * D_)
        else:
            # tree_mask: tree-structured verify step (spec decoding)
            attn = ops.attn_paged_qkv(qkv, Hq, Hkv, kp, vp, pt, start_pos,
                                      self.scale, tree_mask=tree_mask,
                                      longest=context_bound(kv, T))
        if fuse_norm:
            return self._fused_tail(hidden, attn)
        h2, y = self._attended(attn, hidden)
        # residual add fused into the down-projection epilogue
        return self._lin(self._gated(y), self.down_w, "down_w", residual=h2)

    # ------------------------------------------------------------------
    # training path (differentiable; full sequence, no KV cache)
    # ------------------------------------------------------------------
    def forward_train(self, hidden: torch.Tensor, start_pos: int = 0) -> torch.Tensor:
        eps = self.config.rms_norm_eps

        def lin(x_, w, name):
            # training path honors active LoRA adapters too (the inference
            # path routes through self._lin; keep both consistent)
            y = training.linear(x_, w)
            ld = getattr(self, "lora_delta", None)
            if ld is not None:
                d = ld(name, x_)
                if d is not None:
                    y = y + d
            return y

        hidden, x = training.norm(hidden, self.input_norm_w, eps)
        cos, sin = self.rope.get(hidden.device)
        attn = training.rope_attention(lin(x, self.qkv_w, "qkv_w"), cos, sin,
                                       self.Hq, self.Hkv, start_pos, self.scale)
        h2, y = training.add_norm(lin(attn, self.o_w, "o_w"), hidden,
                                  self.post_norm_w, eps)
        m = training.swiglu(training.linear(y, self.gate_up_w))
        return h2 + training.linear(m, self.down_w)

    def forward(self, *args, **kw):
        return self.forward_inference(*args, **kw)


# the step that a span's launch stands for
_LLAMA_STEP = LlamaBlock.forward_inference
