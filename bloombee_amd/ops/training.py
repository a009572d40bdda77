"""Steps of the training path, differentiable: rotary causal attention of whole
sequences on a fused projection, RMS norms around the residual, the gated product,
gradients of frozen projections, prompts added to the first tokens.

Each has a plain torch form, which every tensor can take, and a fused one with
gradient kernels (module _hip_train) for bf16 tensors on the device. The fused form
is an autograd node: it is passed by wherever something watches or replaces the torch
operations themselves (tracing, function transforms, forward-mode, dispatch and
function modes, autocast, tensor subclasses), and gradients that are differentiated
again or taken in batches go through the plain form.
"""
from __future__ import annotations

import importlib
from typing import Tuple

import torch
import torch.nn.functional as F

from bloombee_amd.ops import interface
from bloombee_amd.ops.interface import _fused, _plain

_module = None


def _ext():
    global _module
    if _module is None:
        interface._require_ext()
        try:
            _module = importlib.import_module("bloombee_amd.ops._hip_train")
        except ImportError as e:
            raise RuntimeError(
                "the _hip_train extension is not built but a tensor is on GPU. "
                "Run `python setup.py hip` (PYTORCH_ROCM_ARCH=gfx950). "
                f"Import error was: {e}") from e
    return _module


def _rows(t: torch.Tensor) -> torch.Tensor:
    """t as the kernels read it: contiguous, and 16 bytes at a time."""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _again(*grads: torch.Tensor) -> bool:
    """The gradient is itself recorded, or taken for a batch at once."""
    return torch.is_grad_enabled() or not all(_plain(g) for g in grads)


def _vjp(f, x: torch.Tensor, g: torch.Tensor) -> torch.Tensor:
    """Gradient of f at x through plain operations, differentiable if gradients
    are being recorded."""
    again = torch.is_grad_enabled()
    with torch.enable_grad():
        at = x if again else x.detach().requires_grad_(True)
        return torch.autograd.grad(f(at), at, g, create_graph=again)[0]


# ---------------------------------------------------------------------------
# rotary causal attention
# ---------------------------------------------------------------------------

def _attention(qkv, cos, sin, Hq, Hkv, start, scale):
    B, T, _ = qkv.shape
    X = Hq + 2 * Hkv
    D = qkv.shape[-1] // X
    qkv = qkv.view(B, T, X, D).permute(0, 2, 1, 3)
    q, k, v = qkv.split([Hq, Hkv, Hkv], dim=1)
    pos = torch.arange(start, start + T, device=qkv.device)
    c = cos[pos].view(1, 1, T, D // 2).float()
    s = sin[pos].view(1, 1, T, D // 2).float()

    def rot(t):
        tf = t.float()
        t1, t2 = tf[..., : D // 2], tf[..., D // 2:]
        return torch.cat([t1 * c - t2 * s, t2 * c + t1 * s], -1).to(t.dtype)

    q, k = rot(q), rot(k)
    k = k.repeat_interleave(Hq // Hkv, dim=1)
    v = v.repeat_interleave(Hq // Hkv, dim=1)
    scores = torch.matmul(q.float(), k.float().transpose(-1, -2)) * scale
    mask = torch.ones(T, T, dtype=torch.bool, device=qkv.device).tril()
    scores = scores.masked_fill(~mask, float("-inf"))
    p = torch.softmax(scores, dim=-1)
    attn = torch.matmul(p, v.float()).to(qkv.dtype)
    return attn.permute(0, 2, 1, 3).reshape(B, T, Hq * D)


class _Attention(torch.autograd.Function):
    @staticmethod
    def forward(ctx, qkv, cos, sin, Hq, Hkv, start, scale, keep):
        x = _rows(qkv)
        out, qk, out32, lse = _ext().rope_attention(x, Hq, Hkv, cos, sin, start,
                                                    scale, keep)
        if keep:
            ctx.save_for_backward(qkv, cos, sin, qk, out32, lse)
            ctx.sizes = Hq, Hkv, start, scale
        return out

    @staticmethod
    def backward(ctx, g):
        qkv, cos, sin, qk, out32, lse = ctx.saved_tensors
        Hq, Hkv, start, scale = ctx.sizes
        if _again(g):
            dx = _vjp(lambda x: _attention(x, cos, sin, *ctx.sizes), qkv, g)
        else:
            dx = _ext().rope_attention_grad(
                _rows(g), _rows(qkv), qk, out32, lse, Hq, Hkv, cos, sin,
                start, scale)
        return dx, None, None, None, None, None, None, None


def rope_attention(qkv: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                   Hq: int, Hkv: int, start: int, scale: float) -> torch.Tensor:
    """Causal attention of whole sequences: qkv (B, T, (Hq + 2 Hkv) * D), token t
    at position start + t of the rotation tables -> (B, T, Hq * D)."""
    D = qkv.shape[-1] // (Hq + 2 * Hkv)
    T = qkv.shape[1]
    # head sizes the kernels are compiled for; 64 bits and positions beyond the
    # tables, which torch reports, take the plain form
    if (_fused(qkv) and D in (64, 128) and scale > 0 and Hq % Hkv == 0
            and 0 <= start <= cos.shape[0] - T and T * (Hq // Hkv) < 1 << 30
            and cos.dtype == sin.dtype == torch.float32 and cos.is_contiguous()
            and sin.is_contiguous() and cos.shape == sin.shape
            and cos.shape[1] == D // 2 and cos.device == sin.device == qkv.device):
        keep = torch.is_grad_enabled() and qkv.requires_grad
        return _Attention.apply(qkv, cos, sin, Hq, Hkv, start, scale, keep)
    return _attention(qkv, cos, sin, Hq, Hkv, start, scale)


# ---------------------------------------------------------------------------
# norms around the residual
# ---------------------------------------------------------------------------

def _rms(x, w, eps):
    xf = x.float()
    return (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + eps)
            ).to(x.dtype) * w


def _norm_grad(h, w, eps, gh, gy):
    """Of h and its norm together."""
    if _again(gh, gy):
        return gh + _vjp(lambda t: _rms(t, w, eps), h, gy)
    return _ext().rms_norm_grad(_rows(h), _rows(w), _rows(gy), _rows(gh), eps)


class _Norm(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, eps):
        ctx.save_for_backward(x, w)
        ctx.eps = eps
        return x.view_as(x), interface.rms_norm(_rows(x), _rows(w), eps)

    @staticmethod
    def backward(ctx, gx, gy):
        x, w = ctx.saved_tensors
        return _norm_grad(x, w, ctx.eps, gx, gy), None, None


class _AddNorm(torch.autograd.Function):
    @staticmethod
    def forward(ctx, a, x, w, eps):
        h, y = interface.rms_norm_residual(_rows(a), _rows(x), _rows(w), eps)
        ctx.save_for_backward(h, w)
        ctx.eps = eps
        return h, y

    @staticmethod
    def backward(ctx, gh, gy):
        h, w = ctx.saved_tensors
        dx = _norm_grad(h, w, ctx.eps, gh, gy)
        return dx, dx, None, None


def _norm_sizes(x, w) -> bool:
    H = x.shape[-1]
    return H % 8 == 0 and H <= 16384 and w.shape == (H,)


def norm(x: torch.Tensor, w: torch.Tensor, eps: float,
         ) -> Tuple[torch.Tensor, torch.Tensor]:
    """(x, its RMS norm): going on with the x returned lets the gradients that
    reach it past the norm join in the norm's."""
    if _fused(x, w) and _norm_sizes(x, w):
        return _Norm.apply(x, w, eps)
    return x, _rms(x, w, eps)


def add_norm(a: torch.Tensor, x: torch.Tensor, w: torch.Tensor, eps: float,
             ) -> Tuple[torch.Tensor, torch.Tensor]:
    """(x + a, its RMS norm)."""
    if (_fused(x, w) and _fused(a) and a.shape == x.shape
            and a.device == x.device and _norm_sizes(x, w)):
        return _AddNorm.apply(a, x, w, eps)
    h = x + a
    return h, _rms(h, w, eps)


# ---------------------------------------------------------------------------
# gated product
# ---------------------------------------------------------------------------

def _swiglu(gu):
    g, u = gu.chunk(2, -1)
    return F.silu(g.float()).to(u.dtype) * u


class _SwiGlu(torch.autograd.Function):
    @staticmethod
    def forward(ctx, gu):
        ctx.save_for_backward(gu)
        return interface.swiglu(_rows(gu))

    @staticmethod
    def backward(ctx, gm):
        gu, = ctx.saved_tensors
        if _again(gm):
            return _vjp(_swiglu, gu, gm)
        return _ext().swiglu_grad(_rows(gu), _rows(gm))


def swiglu(gu: torch.Tensor) -> torch.Tensor:
    """silu(gate) * up of (..., [gate | up])."""
    if _fused(gu) and gu.shape[-1] % 16 == 0:
        return _SwiGlu.apply(gu)
    return _swiglu(gu)


# ---------------------------------------------------------------------------
# frozen projections
# ---------------------------------------------------------------------------

def _half_steps(M: int, N: int, K: int) -> bool:
    """Whether the split sum along N, (M, N) @ (N, K), beats the library's GEMM for
    rows of w that come in 32s and not in 64s (gemm_grad.hip). us, split and library,
    N x K:
    28704 x 4096: 1 row 52, 146; 33 57, 163; 128 73, 155; 450 161, 297; 1000 285, 371;
        1200 385, 374
    6176 x 2048: 33 rows 20, 33; 128 25, 33; 200 31, 34
    4128 x 1024: 33 rows 15, 15; 128 20, 19; 300 24, 23
    2080 x 512: any 12 to 24, 9 to 16, where a call is 20 us of the host's time"""
    if N % 64 != 32 or K % 256:
        return False
    tiles = -(-M // 128) * (K // 256)
    return (M <= 128 and N >= K
            or M <= 1024 and N >= 4 * K and K <= 5120 and tiles <= 128)


def _split_gradient(M: int, N: int, K: int) -> bool:
    return _ext().linear_grad_wins(M, N, K) or _half_steps(M, N, K)


class _Linear(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w):
        ctx.save_for_backward(w)
        return interface.linear(x, w)

    @staticmethod
    def backward(ctx, g):
        w, = ctx.saved_tensors
        if (_again(g) or not _plain(w)
                or not _split_gradient(g.numel() // g.shape[-1], *w.shape)):
            return g.matmul(w), None
        rows, w = g.reshape(-1, g.shape[-1]).contiguous(), w.contiguous()
        if rows.data_ptr() % 16 or w.data_ptr() % 16:
            return g.matmul(w), None
        dx = _ext().linear_grad(rows, w, 0)
        return dx.view(*g.shape[:-1], w.shape[1]), None


def linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x @ w^T; w is frozen where the gradient kernel is to take part."""
    if (torch.is_grad_enabled() and x.requires_grad and _fused(x, w)
            and w.dim() == 2 and x.dim() >= 2 and x.shape[-1] == w.shape[1]
            and w.is_contiguous()):
        M = x.numel() // x.shape[-1]
        if (interface.hip_ops.rows_wins(M, *w.shape)
                or _split_gradient(M, *w.shape)):
            return _Linear.apply(x, w)
    return F.linear(x, w)


# ---------------------------------------------------------------------------
# prompts
# ---------------------------------------------------------------------------

def _add_prompts(x, p):
    return torch.cat([x[:, :p.shape[0]] + p.unsqueeze(0), x[:, p.shape[0]:]], 1)


class _AddPrompts(torch.autograd.Function):
    """The gradient of x is the one that arrives, of p the sum of its first rows;
    slices and their concatenation fill, copy and add whole tensors for that (450
    rows of 4096, forward and backward: 68 us, 15)."""

    @staticmethod
    def forward(ctx, x, p):
        ctx.rows = p.shape[0]
        y = x.clone(memory_format=torch.contiguous_format)
        y[:, :ctx.rows] += p
        return y

    @staticmethod
    def backward(ctx, g):
        return g, g[:, :ctx.rows].sum(0)


def add_prompts(x: torch.Tensor, p: torch.Tensor) -> torch.Tensor:
    """x (B, T, H) with p (n, H) added to the first n <= T tokens of every text."""
    if (x.dim() == 3 and p.dim() == 2 and p.shape[0] <= x.shape[1]
            and p.shape[1] == x.shape[2] and p.device == x.device
            and _fused(x) and _fused(p)):
        return _AddPrompts.apply(x, p)
    return _add_prompts(x, p)
