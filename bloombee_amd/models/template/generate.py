"""New-family scaffolding generator (parity: reference models/template/ —
jinja2 codegen from a YAML spec to family config/block/__init__ files,
template/README.md:1-40).

    python -m bloombee_amd.models.template.generate spec_llama.yaml --out DIR
"""
from __future__ import annotations

import argparse
import os
from pathlib import Path

import jinja2
import yaml

CONFIG_T = '''"""{{ Family }} family config — generated by
bloombee_amd.models.template (edit freely; the generator is scaffolding)."""
from __future__ import annotations

from dataclasses import dataclass

from bloombee_amd.models.base import ModelConfig

{{ FAMILY }}_PRESETS = {
{% for name, p in presets.items() %}    "{{ name }}": dict(
{% for k, v in p.items() %}        {{ k }}={{ v }},
{% endfor %}        tie_word_embeddings={{ tie_word_embeddings }},
    ),
{% endfor %}}


@dataclass
class {{ Family }}Config(ModelConfig):
    model_type: str = "{{ family }}"
'''

BLOCK_T = '''"""{{ Family }} server block — generated scaffolding on the shared
gfx950 op layer (see models/llama/block.py for the reference structure)."""
from __future__ import annotations

import math
from typing import Optional

import torch

from bloombee_amd import ops
from bloombee_amd.kv.paged import SessionHandle, context_bound
from bloombee_amd.models.base import ModelConfig
from bloombee_amd.models.llama.block import RopeTables


class {{ Family }}Block(torch.nn.Module):
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
{% if rope %}        self.rope = rope if rope is not None else RopeTables(config)
{% endif %}
        def p(*shape):
            return torch.nn.Parameter(torch.empty(*shape, dtype=dt),
                                      requires_grad=False)

        self.input_norm_w = p(H)
{% if norm == "layernorm" %}        self.input_norm_b = p(H)
{% endif %}        self.qkv_w = p((Hq + 2 * Hkv) * D, H)
        self.o_w = p(H, Hq * D)
        self.post_norm_w = p(H)
{% if norm == "layernorm" %}        self.post_norm_b = p(H)
{% endif %}{% if activation == "swiglu" %}        self.gate_up_w = p(2 * I, H)
{% else %}        self.up_w = p(I, H)
{% endif %}        self.down_w = p(H, I)

    @torch.no_grad()
    def init_random(self, seed: Optional[int] = None):
        s = seed if seed is not None else 1234 + self.layer_index
        dev = self.input_norm_w.device
        gen = torch.Generator(device=dev).manual_seed(s)
        std = 0.02 / math.sqrt(2 * self.config.num_hidden_layers)
        for name, w in self.named_parameters():
            if name.endswith("norm_b"):
                w.zero_()
            elif name.endswith("norm_w"):
                w.fill_(1.0)
            else:
                w.copy_(torch.randn(w.shape, generator=gen, dtype=torch.float32,
                                    device=dev).mul_(std).to(w.dtype))
        return self

    def _norm(self, x, w{% if norm == "layernorm" %}, b{% endif %}):
{% if norm == "layernorm" %}        return ops.layer_norm(x, w, b, self.config.layer_norm_epsilon)
{% else %}        return ops.rms_norm(x, w, self.config.rms_norm_eps)
{% endif %}
    @torch.no_grad()
    def forward_inference(self, hidden: torch.Tensor, kv: SessionHandle,
                          start_pos: torch.Tensor,
                          position_ids=None) -> torch.Tensor:
        B, T, H = hidden.shape
        Hq, Hkv, D = self.Hq, self.Hkv, self.D
        x = self._norm(hidden, self.input_norm_w{% if norm == "layernorm" %}, self.input_norm_b{% endif %})
        qkv = ops.linear(x, self.qkv_w)
        kp = kv.k_pages(self.layer_index)
        vp = kv.v_pages(self.layer_index)
        pt = kv.page_table()
{% if rope %}        cos, sin = self.rope.get(hidden.device)
        ops.rope_kv_write_(qkv, Hq, Hkv, cos, sin, position_ids, kp, vp, pt,
                           start_pos)
{% else %}        q = qkv[..., :Hq * D].view(B, T, Hq, D).permute(0, 2, 1, 3).contiguous()
        k = qkv[..., Hq * D:(Hq + Hkv) * D].view(B, T, Hkv, D).permute(0, 2, 1, 3).contiguous()
        v = qkv[..., (Hq + Hkv) * D:].view(B, T, Hkv, D).permute(0, 2, 1, 3).contiguous()
        ops.kv_write(k, v, kp, vp, pt, start_pos)
{% endif %}        attn = ops.attn_paged_qkv(qkv, Hq, Hkv, kp, vp, pt, start_pos, self.scale,
                                  longest=context_bound(kv, T))
        a = ops.linear(attn, self.o_w)
        h = hidden + a
        y = self._norm(h, self.post_norm_w{% if norm == "layernorm" %}, self.post_norm_b{% endif %})
{% if activation == "swiglu" %}        m = ops.linear(ops.swiglu(ops.linear(y, self.gate_up_w)), self.down_w)
{% else %}        m = ops.linear(ops.gelu_tanh(ops.linear(y, self.up_w)), self.down_w)
{% endif %}        return h + m

    def forward_train(self, hidden: torch.Tensor, start_pos: int = 0):
        raise NotImplementedError(
            "generated scaffolding: fill in the eager training path "
            "(copy the structure from models/llama/block.py forward_train)")

    def forward(self, *a, **k):
        return self.forward_inference(*a, **k)
'''

INIT_T = '''from bloombee_amd.models.base import FamilyEntry, register_model_family
from bloombee_amd.models.llama.model import (DistributedLlamaForCausalLM,
                                             DistributedLlamaModel)

from .block import {{ Family }}Block
from .config import {{ FAMILY }}_PRESETS, {{ Family }}Config

register_model_family(
    "{{ family }}",
    FamilyEntry(config_cls={{ Family }}Config, block_cls={{ Family }}Block,
                model_cls=DistributedLlamaModel,
                causal_lm_cls=DistributedLlamaForCausalLM,
                presets={{ FAMILY }}_PRESETS),
)
'''


def generate_family(spec_path: str, out_dir: str) -> Path:
    spec = yaml.safe_load(Path(spec_path).read_text())
    family = spec["family"]
    env = jinja2.Environment(keep_trailing_newline=True)
    ctx = {
        "family": family,
        "Family": family.capitalize(),
        "FAMILY": family.upper(),
        "norm": spec.get("norm", "rms"),
        "activation": spec.get("activation", "swiglu"),
        "rope": bool(spec.get("rope", True)),
        "tie_word_embeddings": bool(spec.get("tie_word_embeddings", False)),
        "presets": spec.get("presets", {}),
    }
    d = Path(out_dir) / family
    d.mkdir(parents=True, exist_ok=True)
    (d / "config.py").write_text(env.from_string(CONFIG_T).render(**ctx))
    (d / "block.py").write_text(env.from_string(BLOCK_T).render(**ctx))
    (d / "__init__.py").write_text(env.from_string(INIT_T).render(**ctx))
    return d


def main():
    ap = argparse.ArgumentParser(description=__doc__)
    ap.add_argument("spec")
    ap.add_argument("--out", default=".")
    args = ap.parse_args()
    d = generate_family(args.spec, args.out)
    print(f"generated family package at {d}")


if __name__ == "__main__":
    main()
