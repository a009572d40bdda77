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


@functools.lru_cache(256)
def _fits(*sizes: int) -> bool:
    return _ext().span_fits(*sizes)


def span_fits(hidden: torch.Tensor, I: int, Hq: int, k_pages: torch.Tensor) -> bool:
    """Whether layers of these sizes may be run in one launch: what rules out most steps,
    to be asked ahead of every layer's tensors (22 layers that do not fit: 66 of an eager
    step's 954 us of the host where they were walked first)."""
    B, T, H = hidden.shape
    return (T == 1 and hidden.is_cuda and hidden.dtype == torch.bfloat16
            and hidden.device.index == torch.cuda.current_device()
            and _whole_device(hidden.device.index) and k_pages.dim() == 4
            and _fits(B, H, I, Hq, k_pages.shape[1], k_pages.shape[3],
                      k_pages.shape[2]))


def decode_span(hidden: torch.Tensor, weights: List[torch.Tensor], Hq: int, cos, sin,
                position_ids: Optional[torch.Tensor], start_pos: torch.Tensor,
                page_table: torch.Tensor, eps: float,
                scale: float) -> Optional[torch.Tensor]:
    """hidden (B, 1, H) through layers of eight tensors each in weights: qkv, o, gate_up
    and down projections, q and k head norms (both empty: none), pages of keys and of
    values. The new tokens' keys and values are in the pages afterwards. Callers have
    asked span_fits; None where the tensors are others than these sizes' after all."""
    pos = position_ids.int().contiguous() if position_ids is not None else None
    return _ext().decode_span_if(hidden.contiguous(), weights, Hq, cos, sin, pos,
                                 start_pos.int().contiguous(), page_table, eps, scale)
