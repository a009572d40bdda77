"""Row kernels whose loads run ahead, at the edges of their chunks: residual sums of
rows that end within a chunk or a vector, router products of partial tiles."""
import pytest
import torch

from bloombee_amd.ops import ragged

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def draw(*shape, seed=0):
    gen = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=gen).to(DEV)


@pytest.mark.parametrize("N", [3, 257])          # 1024 threads a row, 256
@pytest.mark.parametrize("W,cols", [(4, 64), (1020, 1024), (4096, 4096), (4100, 4160),
                                    (4098, 4098), (9000, 9024)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("groups,shift", [(1, 0), (2, 0), (1, 1)])
def test_plain_residual_sum(N, W, cols, dt, groups, shift):
    x, parts = draw(N, W, seed=1), draw(1, N, W, seed=2).to(dt)
    w = draw(W + shift, seed=3)[shift:]          # weights that are not aligned
    want = x.double() + parts[0].double()
    got = x.clone()
    h = ragged.residual_norm(got, ragged.Pending(parts), w, groups, 1e-5, cols)
    # one 32-bit sum
    assert bool(((got.double() - want).abs() <= 2.0 ** -23 * want.abs()).all())
    g = want.view(N, groups, W // groups)
    n = g * torch.rsqrt(g.pow(2).mean(-1, keepdim=True) + 1e-5)
    n = n.view(N, W) * w.double()
    # one rounding to bf16 behind 32-bit sums
    assert bool(((h[:, :W].double() - n).abs() <= 2.01 * 2.0 ** -9 * n.abs()).all())
    assert bool((h[:, W:] == 0).all())
    x2 = x.clone()
    h2 = ragged.sum_norm(x2, parts, None, w, 0.5, 1e-5, cols, torch.bfloat16)
    want = 0.5 * x.double() + parts[0].double()
    n = want * torch.rsqrt(want.pow(2).mean(-1, keepdim=True) + 1e-5) * w.double()
    assert bool(((x2.double() - n).abs() <= 1e-5 * n.abs() + 1e-6).all())
    assert torch.equal(h2[:, :W], x2.bfloat16()) and bool((h2[:, W:] == 0).all())


@pytest.mark.parametrize("N", [3, 257])
@pytest.mark.parametrize("W,cols", [(8, 8), (1024, 1024), (1028, 6016), (8192, 8192),
                                    (8196, 8256), (16384, 16384), (16388, 20480)])
@pytest.mark.parametrize("splits,biased", [(0, False), (1, False), (1, True), (3, True)])
def test_norms_of_rows_in_registers(N, W, cols, splits, biased):
    """Rows that fill a thread's pieces and one vector more; without parts the residual
    stays as it is."""
    x, w = draw(N, W, seed=1), draw(W, seed=3)
    x[-1, W // 2] = float("inf")                  # its row is not a number there
    parts = draw(max(splits, 1), N, W, seed=2).bfloat16()
    bias = draw(W, seed=4) if biased else None
    pending = ragged.Pending(parts, keep=0.5, bias=bias) if splits else None
    got = x.clone()
    h = ragged.residual_norm(got, pending, w, 1, 1e-5, cols)
    want = 0.5 * x.double() + parts.double().sum(0) if splits else x.double()
    if splits:
        more = bias.double() if biased else torch.zeros_like(w).double()
        want = want + more
        # a rounding of 32 bits a term
        bound = 2.0 ** -22 * (x.double().abs() + parts.double().abs().sum(0) + more.abs())
        assert bool((((got.double() - want).abs() <= bound) | want.isinf()).all())
    else:
        assert torch.equal(got, x)
    n = want * torch.rsqrt(want.pow(2).mean(-1, keepdim=True) + 1e-5) * w.double()
    # one rounding to bf16 behind 32-bit sums, whose terms may cancel
    near = (h[:, :W].double() - n).abs() <= 2.01 * 2.0 ** -9 * n.abs() + 1e-5
    assert bool((near | n.isnan()).all())
    assert torch.equal(h[:, :W].isnan(), n.isnan()) and bool((h[:, W:] == 0).all())


@pytest.mark.parametrize("M,N,K", [(1, 1, 32), (16, 16, 96), (17, 17, 256),
                                   (33, 80, 288), (15, 15, 4128)])
def test_router_tiles(M, N, K):
    a, w = draw(M, K, seed=1).bfloat16(), draw(N, K, seed=2).bfloat16()
    got = ragged._ext().router_gemm(a, w)[0]
    want = a.double() @ w.double().T
    # products of bf16 are exact in 32 bits, sums round K times at most
    bound = K * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)
    assert bool(((got.double() - want).abs() <= bound).all())
