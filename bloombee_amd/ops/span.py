"""A decode step of a span of dense decoder layers in one launch
(ops/hip/decode_span.hip): BlockStack takes it where it wins, layer by layer elsewhere."""
from __future__ import annotations

import functools
import importlib
from typing import List, Optional

import torch

from bloombee_amd.ops import interface

_hip_span = None


def _ext():
    global _hip_span
    if _hip_span is None:
        interface._require_ext()
        _hip_span = importlib.import_module("bloombee_amd.ops._hip_span")
    return _hip_span


@functools.lru_cache(None)
def _whole_device(index: int) -> bool:
    """As many compute units as the kernel has slots."""
    return torch.cuda.get_device_properties(index).multi_processor_count >= 256


def decode_span(hidden: torch.Tensor, weights: List[torch.Tensor], Hq: int, cos, sin,
                position_ids: Optional[torch.Tensor], start_pos: torch.Tensor,
                page_table: torch.Tensor, eps: float,
                scale: float) -> Optional[torch.Tensor]:
    """hidden (B, 1, H) through layers of eight tensors each in weights: qkv, o, gate_up
    and down projections, q and k head norms (both empty: none), pages of keys and of
    values. The new tokens' keys and values are in the pages afterwards. None where the
    layers are to be run one by one."""
    B, T, H = hidden.shape
    if (T != 1 or not hidden.is_cuda or hidden.dtype != torch.bfloat16
            or hidden.device.index != torch.cuda.current_device()
            or not _whole_device(hidden.device.index)):
        return None
    pos = position_ids.int().contiguous() if position_ids is not None else None
    args = (hidden.contiguous(), weights, Hq, cos, sin, pos, start_pos.int().contiguous(),
            page_table)
    ext = _ext()
    if not ext.span_takes(*args):
        return None
    return ext.decode_span(*args, eps, scale)
