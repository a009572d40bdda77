"""Products of some dozen rows to a thousand on the tiles of gemm_rows.hip."""
import pytest
import torch

from bloombee_amd import ops
from bloombee_amd.ops import training

pytestmark = pytest.mark.gpu
DEV = "cuda"


def draw(*shape, seed, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * scale).bfloat16()


def close(got, want, terms):
    """The result's rounding, 2^-9, and 32-bit sums of `terms` (the sum of the
    products' magnitudes) in any order."""
    return bool(((got.double() - want).abs()
                 <= 2.0 ** -8 * want.abs() + 2.0 ** -20 * terms + 1e-30).all())


# (rows, columns, K): every tile, unsplit and split; one row, strip or column short of a
# tile or past it; fewer steps than buffers, as many, more
SIZES = [(33, 8, 256), (65, 136, 320), (97, 248, 448), (129, 4096, 1024),
         (192, 1032, 704), (193, 28672, 256), (200, 6144, 1088), (256, 10240, 512),
         (333, 4096, 4096), (450, 4096, 5120), (512, 8192, 1536), (617, 6208, 576),
         (768, 6144, 1536), (1000, 1024, 3072), (1025, 4104, 448), (1400, 4096, 1024),
         (193, 42568, 256), (138, 33360, 256), (167, 33064, 320), (203, 32960, 256),
         (333, 28672, 512), (1891, 8, 7168), (1650, 8, 7104), (300, 33000, 704)]


GATED = [(33, 8, 256), (97, 1000, 320), (200, 14336, 256), (333, 14336, 448),
         (450, 56, 4096), (617, 4096, 384), (1000, 8192, 512), (64, 120, 576),
         (194, 21360, 256), (194, 21360, 320), (155, 17032, 256), (171, 19000, 256), (222, 16880, 256),
         (226, 13024, 256), (131, 11224, 256), (109, 8312, 256), (65, 8912, 256)]


@pytest.mark.parametrize("M,N,K", SIZES)
def test_product(M, N, K):
    x, w = draw(M, K, seed=1), draw(N, K, seed=2, scale=K ** -0.5)
    r, b = draw(M, N, seed=3), draw(N, seed=4)
    assert ops.hip_ops.rows_wins(M, N, K)
    want = x.double() @ w.double().T
    terms = x.double().abs() @ w.double().abs().T
    assert close(ops.linear(x, w), want, terms)
    more = want + r.double() + b.double()
    assert close(ops.linear(x, w, residual=r, bias=b), more,
                 terms + r.double().abs() + b.double().abs())


def test_tiles_are_reached():
    plans = {ops.hip_ops.rows_plan(M, N, K, False) for M, N, K in SIZES}
    assert {t for t, _ in plans} == set(range(10)) and len({s for _, s in plans}) >= 3
    plans = {ops.hip_ops.rows_plan(M, 2 * F, K, True) for M, F, K in GATED}
    assert plans == {(t, 1) for t in range(9)}


@pytest.mark.parametrize("M,F,K", GATED)
def test_gated(M, F, K):
    x, w = draw(M, K, seed=1), draw(2 * F, K, seed=2, scale=K ** -0.5)
    g, u = (x.double() @ w.double().T).chunk(2, -1)
    want = torch.nn.functional.silu(g) * u
    got = ops.hip_ops.gemm_rows_swiglu(x, w)
    # sums of 32 bits within 2^-20 of their terms, hardware exponential and reciprocal
    tol = (x.double().abs() @ w.double().abs().T).chunk(2, -1)
    assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs()
                 + 2.0 ** -19 * (tol[0] * u.abs() + tol[1] * g.abs()) + 1e-30).all())
    y = ops.linear_gated(x, w)
    # where it is two steps, gate and up are rounded, 2^-9 of each
    assert bool(((y.double() - want).abs() <= 2.0 ** -8 * want.abs()
                 + 2.0 ** -8 * (g.abs() + 1) * u.abs() + 1e-6).all())


@pytest.mark.parametrize("M,F,K", [(257, 20480, 256), (300, 28672, 320), (320, 18432, 448),
                                   (617, 11088, 1024), (640, 14336, 256), (601, 28000, 576)])
def test_gated_on_the_tall_tile(M, F, K):
    """One row tile, whose W passes the caches, and two."""
    assert ops.hip_ops.rows_tall(M, 2 * F, K)
    test_gated(M, F, K)


FEW = [(1, 28672, 1024), (9, 5120, 13824), (16, 4096, 14336), (17, 28672, 1280),
       (31, 576, 9216), (32, 8192, 8192), (32, 6144, 4096), (5, 192, 14336)]


@pytest.mark.parametrize("M,N,K", FEW)
def test_few_rows(M, N, K):
    x, w = draw(M, K, seed=1), draw(N, K, seed=2, scale=K ** -0.5)
    r, b = draw(M, N, seed=3), draw(N, seed=4)
    want = x.double() @ w.double().T
    terms = x.double().abs() @ w.double().abs().T
    assert ops.hip_ops.few_sums(M, N, K)
    assert close(ops.linear(x, w), want, terms)
    assert close(ops.linear(x, w, residual=r, bias=b), want + r.double() + b.double(),
                 terms + r.double().abs() + b.double().abs())


@pytest.mark.parametrize("M,N,K", [(17, 26304, 1024), (18, 12288, 1280), (25, 28672, 4096),
                                   (32, 27648, 1280), (17, 57344, 1024), (31, 98304, 1024)])
def test_few_rows_gated(M, N, K):
    """The rows' norm, folded into w, rides along."""
    x, w = draw(M, K, seed=1, scale=3.0), draw(N, K, seed=2, scale=K ** -0.5)
    x[0] *= 1e-3      # where eps counts
    assert ops.hip_ops.few_swiglu(M, N, K)
    y = x.double()
    r = (y.square().mean(-1, keepdim=True) + 1e-5).rsqrt()
    g, u = ((y @ w.double().T) * r).chunk(2, -1)
    want = torch.nn.functional.silu(g) * u
    got = ops.linear_swiglu(x, w, 1e-5)
    tol = ((y.abs() @ w.double().abs().T) * r).chunk(2, -1)
    # sums and root within 2^-20 of their terms, hardware exponential and reciprocal
    assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs()
                 + 2.0 ** -18 * (tol[0] * (u.abs() + 1) + tol[1] * (g.abs() + 1))).all())


@pytest.mark.parametrize("N,K,width", [
    (64, 512, 32), (8192, 256, 32), (8256, 512, 64), (16384, 768, 64), (16448, 256, 96),
    (24576, 1024, 96), (24640, 512, 128), (32768, 256, 128), (32832, 512, 160),
    (40960, 256, 160), (41024, 256, 96)])
@pytest.mark.parametrize("M", [1, 9, 32])
def test_widths_of_few_rows(M, N, K, width):
    """One tile and strip short of a round of workgroups, or past it; fewer stages than
    buffers."""
    test_few_rows_gated(M, N, K)
    assert ops.hip_ops.few_width(N) == width


@pytest.mark.parametrize("Hq,Hkv,D,K,width", [
    (4, 2, 32, 1024, 32), (61, 1, 128, 1024, 32), (28, 6, 256, 1024, 64),
    (200, 28, 96, 1024, 96), (1000, 10, 32, 1024, 128), (260, 2, 128, 1280, 160)])
@pytest.mark.parametrize("B,T", [(1, 1), (3, 3), (32, 1), (2, 11)])
@pytest.mark.parametrize("placed", [False, True])
def test_turned_projections(Hq, Hkv, D, K, width, B, T, placed):
    """Tiles that end within a head or take several; rows short of a strip."""
    N = (Hq + 2 * Hkv) * D
    assert ops.hip_ops.few_rope(B * T, N, K) and ops.hip_ops.few_width(N) == width
    x, w = draw(B, T, K, seed=1), draw(N, K, seed=2, scale=K ** -0.5)
    P, start = 16, torch.arange(B, device=DEV, dtype=torch.int32) * 7 + 13
    maxp = (7 * B + 13 + T) // P + 1
    table = torch.randperm(B * maxp, device=DEV).int().view(B, maxp)
    kp = draw(B * maxp, Hkv, P, D, seed=3)
    vp = draw(B * maxp, Hkv, D, P, seed=4)
    pos = torch.randint(0, 400, (B, T), device=DEV).int() if placed else None
    cos, sin = (t.to(DEV) for t in ops.rope_cos_sin(D, 512))
    y = x.double()
    z = (y * (y.square().mean(-1, keepdim=True) + 1e-5).rsqrt()) @ w.double().T
    want, kw, vw = z.float().cpu(), kp.float().cpu(), vp.float().cpu()
    ops.rope_kv_write_(want, Hq, Hkv, cos.cpu(), sin.cpu(),
                       None if pos is None else pos.cpu(), kw, vw, table.cpu(),
                       start.cpu())
    got = ops.linear_rope_kv(x, w, 1e-5, Hq, Hkv, cos, sin, pos, kp, vp, table, start)
    # one rounding of 32-bit sums, 2^-9 of a value; turns and root within 2^-18 of terms
    for a, b in ((got[..., :Hq * D], want[..., :Hq * D]), (kp, kw), (vp, vw)):
        assert bool(((a.float().cpu() - b).abs() <= 2.0 ** -8 * b.abs() + 1e-4).all())


@pytest.mark.parametrize("K", [256, 320, 448, 512, 576, 4096])
@pytest.mark.parametrize("M", [40, 64])
def test_one_row_tile(M, K):
    """Each XCD begins with another stage of K, of fewer than eight too."""
    N = 8192
    x, w = draw(M, K, seed=1), draw(N, K, seed=2, scale=K ** -0.5)
    assert ops.hip_ops.rows_plan(M, N, K, False)[1] == 1 or K == 4096
    want = x.double() @ w.double().T
    terms = x.double().abs() @ w.double().abs().T
    assert close(ops.hip_ops.gemm_rows(x, w, None, None), want, terms)
    g, u = want.chunk(2, -1)
    tol = terms.chunk(2, -1)
    got = ops.hip_ops.gemm_rows_swiglu(x, w)
    want = torch.nn.functional.silu(g) * u
    assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs()
                 + 2.0 ** -19 * (tol[0] * u.abs() + tol[1] * g.abs()) + 1e-30).all())


@pytest.mark.parametrize("M,N,K,plan", [
    (1, 4160, 512, (32, 1)), (3, 8192, 512, (32, 1)), (7, 16320, 1024, (64, 1)),
    (1, 20480, 1024, (96, 1)), (5, 28672, 1024, (128, 1)), (9, 36864, 1024, (160, 1)),
    (8, 2560, 8448, (64, 6)), (13, 1024, 4864, (64, 9)), (17, 2048, 4096, (64, 8)),
    (32, 6144, 4096, (32, 1))])
def test_few_rows_by_their_plan(M, N, K, plan):
    """Every width unsplit, and the splits of few columns."""
    assert ops.hip_ops.few_wins(M, N, K) and ops.hip_ops.few_plan(M, N, K) == plan
    x, w = draw(M, K, seed=1), draw(N, K, seed=2, scale=K ** -0.5)
    r, b = draw(M, N, seed=3), draw(N, seed=4)
    want = x.double() @ w.double().T
    terms = x.double().abs() @ w.double().abs().T
    assert close(ops.linear(x, w), want, terms)
    assert close(ops.linear(x, w, residual=r, bias=b), want + r.double() + b.double(),
                 terms + r.double().abs() + b.double().abs())


@pytest.mark.parametrize("M,F,up,cols,K", [
    (33, 8, 8, 64, 256), (65, 1000, 1024, 1088, 320), (200, 4096, 4100, 4096, 256),
    (333, 712, 715, 768, 576), (617, 1400, 1400, 1408, 384), (194, 21360, 21376, 21504, 256)])
@pytest.mark.parametrize("bias", [False, True])
def test_clamped(M, F, up, cols, K, bias):
    """Activations that end within a tile, columns of zeros behind them."""
    from bloombee_amd.ops import ragged
    x, w = draw(M, K, seed=1), draw(up + F, K, seed=2, scale=K ** -0.5)
    b = ((torch.randn(F, device=DEV), torch.randn(F, device=DEV)) if bias
         else (None, None))
    g, u = (x.double() @ w[o:o + F].double().T + (0 if v is None else v.double())
            for o, v in zip((0, up), b))
    g, u = g.clamp(max=1.5), u.clamp(-1.5, 1.5)
    want = g * torch.sigmoid(1.702 * g) * (u + 1)
    got = ops.hip_ops.gemm_rows_glu(x, w, up, F, cols, *b, 1.5, 1.702)
    # a sum is off by 2^-20 of its terms, their product by as much of both
    tol = (x.double().abs() @ w[:F].double().abs().T,
           x.double().abs() @ w[up:].double().abs().T)
    assert bool(((got[:, :F].double() - want).abs() <= 2.0 ** -8 * want.abs()
                 + 2.0 ** -18 * (tol[0] * 2.5 + tol[1] * g.abs() + 1)).all())
    assert got.shape == (M, cols) and not got[:, F:].any()
    y = ragged.linear_glu(x, w, up, F, *b, 1.5, 1.702, cols, torch.bfloat16)
    # where it is two steps, gate and up are rounded, 2^-9 of each
    assert bool(((y[:, :F].double() - want).abs() <= 2.0 ** -8 * want.abs()
                 + 2.0 ** -7 * (g.abs() + 1) * 2.5).all()) and not y[:, F:].any()


# (rows, rows of w, columns): every tile, one row short of it or past it, fewer steps
# than buffers and more
GRADS = [(1, 64, 256), (63, 128, 512), (65, 448, 4096), (134, 128, 11520),
         (202, 320, 11520), (284, 1728, 11520), (643, 64, 11264), (643, 128, 11264),
         (643, 192, 11264), (643, 256, 11264), (520, 192, 13312), (450, 4096, 14336),
         (193, 15168, 11008), (450, 6144, 4096), (333, 28672, 1024), (1999, 4096, 4096)]


@pytest.mark.parametrize("M,N,K", GRADS)
@pytest.mark.parametrize("splits", [0, 1, 5])
def test_gradient(M, N, K, splits):
    g, w = draw(M, N, seed=1), draw(N, K, seed=2, scale=N ** -0.5)
    got = training._ext().linear_grad(g, w, splits)
    # in blocks: the magnitudes in 64 bits are large
    for r in range(0, M, 500):
        a = g[r:r + 500].double()
        assert close(got[r:r + 500], a @ w.double(), a.abs() @ w.double().abs())


def test_gradient_tiles_are_reached():
    plans = {training._ext().linear_grad_plan(*s) for s in GRADS}
    assert {t for t, _ in plans} == set(range(7)) and len({s for _, s in plans}) >= 3


def test_not_finite():
    """Infinities and NaN stay in their rows and columns."""
    M, N, K = 100, 640, 512
    x, w = draw(M, K, seed=1), draw(N, K, seed=2)
    x[7, 3], x[99, 511], w[5, 0] = float("inf"), float("nan"), float("-inf")
    want = x.float() @ w.float().T
    got = ops.linear(x, w).float()
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isinf(), want.isinf())
    some = want.isfinite()
    assert torch.allclose(got[some], want[some], rtol=2.0 ** -7, atol=1e-3)


def test_addends_are_torchs():
    """What is added keeps its tangent and broadcasts, or is refused, as torch has it."""
    import torch.autograd.forward_ad as fwd
    M, N, K = 64, 64, 256
    x, w = draw(M, K, seed=1), draw(N, K, seed=2, scale=K ** -0.5)
    r, t = draw(M, N, seed=3), draw(M, N, seed=4)
    assert ops.hip_ops.rows_wins(M, N, K)
    with fwd.dual_level():
        y = fwd.unpack_dual(ops.linear(x, w, residual=fwd.make_dual(r, t)))
        assert torch.equal(y.tangent, t)
        y = fwd.unpack_dual(ops.linear(x, w, bias=fwd.make_dual(r[0], t[0])))
        assert torch.equal(y.tangent, t[0].expand(M, N))
    rows = draw(M, 1, seed=5)                # one value a row
    assert close(ops.linear(x, w, bias=rows), x.double() @ w.double().T + rows.double(),
                 x.double().abs() @ w.double().abs().T + rows.double().abs())
    apart = draw(2, M, N // 2, seed=6).transpose(0, 1)   # no view of (M, N)
    with pytest.raises(RuntimeError):
        ops.linear(x, w, residual=apart)
    with pytest.raises(RuntimeError):
        ops.linear(x, w[:32], bias=rows[:32])
    # any other layout of the right shape, and any shape of the right values
    for res in (draw(N, M, seed=8).T, draw(M * N, seed=9), draw(M, 2 * N, seed=9)[:, N:]):
        assert close(ops.linear(x, w, residual=res),
                     x.double() @ w.double().T + res.reshape(M, N).double(),
                     x.double().abs() @ w.double().abs().T + res.reshape(M, N).double().abs())


@pytest.mark.parametrize("M", [1, 8, 20, 64])
@pytest.mark.parametrize("K", [256, 2048])
def test_weights_without_rows(M, K):
    from bloombee_amd.ops import ragged
    x, w = draw(M, K, seed=1), draw(0, K, seed=2)
    assert ops.linear(x, w).shape == (M, 0)
    assert ops.hip_ops.gemm_stream(x[:32], w, None, None, -1.0).shape == (min(M, 32), 0)
    if K == 2048 and M <= 32:
        with pytest.raises(RuntimeError):      # refused, no division by its columns
            ops.hip_ops.gemm_skinny(x, w, None, None, 0, None, 0.0, None, None, 0)
        with pytest.raises(RuntimeError):
            ragged._ext().gemm_parts(x, w, 0)
    x.requires_grad_(True)
    dx, = torch.autograd.grad(training.linear(x, w).sum(), x)
    assert dx.shape == x.shape and not dx.any()
    torch.cuda.synchronize()
    assert not draw(M, K, seed=1).isnan().any()     # no error is left for the next call


def test_sizes_are_asked_first(monkeypatch):
    """Products that the rules leave to others do not pay for a look at their tensors."""
    from bloombee_amd.ops import interface, ragged

    def look(*tensors):
        raise AssertionError("looked at")
    monkeypatch.setattr(interface, "_readable", look)
    b = torch.zeros(1024, device=DEV)
    for M in (1, 8, 32):       # a decode step's rows
        x, w = draw(M, 256, seed=1), draw(2048, 256, seed=2)
        ragged.linear_glu(x, w, 1024, 1024, b, b, 1.5, 1.702, 1024, torch.bfloat16)
        ops.linear_gated(x, w)
        ops.linear(x, w)
    x, w = draw(64, 264, seed=1), draw(2048, 264, seed=2)     # K % 64
    ops.linear_gated(x, w)
    with pytest.raises(AssertionError):
        ops.linear(draw(64, 256, seed=1), draw(2048, 256, seed=2))


def test_views():
    """Rows at any address and of any stride, weights that do not begin at 16 bytes."""
    M, N, K = 64, 256, 320
    flat = draw(M * K + 1, seed=1)
    w = draw(N, K, seed=2)
    for x in (flat[1:].view(M, K), draw(M, 2 * K, seed=3)[:, :K],
              draw(K, M, seed=4).T, draw(2, M // 2, K, seed=5)):
        want = x.double() @ w.double().T
        terms = x.double().abs() @ w.double().abs().T
        assert close(ops.linear(x, w), want, terms)
    odd = draw(N * K + 1, seed=6)[1:].view(N, K)
    x = draw(M, K, seed=7)
    assert close(ops.linear(x, odd), x.double() @ odd.double().T,
                 x.double().abs() @ odd.double().abs().T)


def test_places_of_32_bits():
    """Rows too long for a tile's places are left to the kernels that had them."""
    assert ops.hip_ops.few_sums(1, 64, (1 << 20) - 128)
    assert not ops.hip_ops.few_sums(1, 64, 1 << 20)
    assert not ops.hip_ops.rows_wins(33, 64, 1 << 20)
    assert not ops.hip_ops.rows_swiglu_wins(33, 64, 1 << 20)


def test_recorded_and_replayed():
    """Gradients reach x through linear; a captured product gives the eager one's bits
    on every replay."""
    M, N, K = 100, 1024, 1024
    x, w = draw(M, K, seed=1).requires_grad_(True), draw(N, K, seed=2)
    g = draw(M, N, seed=3)
    for f in (ops.linear, training.linear):
        dx, = torch.autograd.grad(f(x, w), x, g)
        assert close(dx, g.double() @ w.double(), g.double().abs() @ w.double().abs())
    at = x.detach().clone()
    ops.linear(at, w)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.linear(at, w)
    for seed in (4, 5, 6):
        at.copy_(draw(M, K, seed=seed))
        graph.replay()
        assert torch.equal(out, ops.linear(at, w))


@pytest.mark.parametrize("M,N,K", [(33, 4096, 4096), (64, 512, 1024), (97, 4096, 1536),
                                   (250, 5120, 4096), (40, 8192, 8192), (33, 16384, 1024),
                                   (512, 1024, 512), (33, 1032, 2048)])
def test_fold_with_norm(M, N, K):
    """The fold of a split product that makes a row's norm too, and products unsplit."""
    x, w = draw(M, K, seed=1), draw(N, K, seed=2, scale=K ** -0.5)
    r, nw = draw(M, N, seed=3), draw(N, seed=4)
    h, y = ops.hip_ops.gemm_rows_norm(x, w, r, nw, 1e-5)
    xd, wd = x.double(), w.double()
    want = xd @ wd.t() + r.double()
    # unsplit, the product is rounded ahead of the residual
    assert close(h, want, xd.abs() @ wd.abs().t()
                 + 2.0 ** 12 * (want - r.double()).abs())
    hd = h.double()
    norm = hd * torch.rsqrt(hd.pow(2).mean(-1, keepdim=True) + 1e-5) * nw.double()
    assert close(y, norm, norm.abs() * 2.0 ** 6)


@pytest.mark.parametrize("B,T,Hq,Hkv,D,P,K,pos", [
    (33, 1, 16, 4, 128, 32, 2048, False), (97, 1, 32, 8, 128, 32, 4096, True),
    (20, 4, 8, 8, 64, 16, 1024, False), (40, 1, 4, 1, 256, 8, 2048, True),
    (35, 2, 6, 3, 32, 32, 4096, False), (12, 5, 16, 4, 128, 32, 2048, False),
    (300, 1, 8, 2, 96, 16, 2048, False), (700, 1, 8, 2, 64, 32, 512, False)])
def test_fold_with_rotation(B, T, Hq, Hkv, D, P, K, pos):
    """The fold of a split product that turns queries and keys and fills the pages, and
    the steps apart where it does not."""
    M, N, half, maxp = B * T, (Hq + 2 * Hkv) * D, D // 2, 4
    x, w = draw(B, T, K, seed=1), draw(N, K, seed=2, scale=K ** -0.5)
    angle = torch.arange(200, device=DEV)[:, None] * torch.rand(half, device=DEV)
    cos, sin = angle.cos(), angle.sin()
    start = (torch.arange(B, device=DEV) * 7 % (P * maxp - T)).int()
    table = torch.randperm(B * maxp, device=DEV).int().view(B, maxp)
    at = start[:, None].long() + torch.arange(T, device=DEV)
    ids = (at * 3 % 150).int() if pos else None
    kp = draw(B * maxp, Hkv, P, D, seed=5)
    vp = draw(B * maxp, Hkv, D, P, seed=6)
    kept_k, kept_v = kp.clone(), vp.clone()
    got = ops.linear_rope_kv_rows(x, w, Hq, Hkv, cos, sin, ids, kp, vp, table, start)
    xd, wd = x.view(M, K).double(), w.double()
    flat, terms = xd @ wd.t(), xd.abs() @ wd.abs().t()
    # apart, the product is rounded ahead of the rotation
    terms = (terms + 2.0 ** 12 * flat.abs()).view(B, T, -1, D)
    y = flat.view(B, T, -1, D)
    where = (ids if pos else at).long()
    c, s = cos.double()[where][:, :, None], sin.double()[where][:, :, None]
    turned = torch.cat([y[..., :half] * c - y[..., half:] * s,
                        y[..., half:] * c + y[..., :half] * s], -1)
    both = terms[..., :half] + terms[..., half:]
    both = torch.cat([both, both], -1)
    q = got.view(B, T, -1, D)[:, :, :Hq]
    assert close(q, turned[:, :, :Hq], both[:, :, :Hq])
    page = table.long().gather(1, at // P)
    k = kp[page, :, at % P]
    assert close(k, turned[:, :, Hq:Hq + Hkv], both[:, :, Hq:Hq + Hkv])
    v = vp[page, :, :, at % P]
    assert close(v, y[:, :, Hq + Hkv:], terms[:, :, Hq + Hkv:])
    kept_k[page, :, at % P] = k
    kept_v[page, :, :, at % P] = v
    assert torch.equal(kp, kept_k) and torch.equal(vp, kept_v)


@pytest.mark.parametrize("N,K", [(64, 512), (576, 4096), (8256, 2048), (4096, 4096),
                                 (40960, 1024), (28672, 640), (192, 16384), (33024, 512)])
def test_parts_of_few_rows(N, K):
    """Partial sums in 32 bits of any width and number of splits; W that does not begin
    at 16 bytes."""
    from bloombee_amd.ops import ragged
    w = draw(N, K, seed=2, scale=K ** -0.5)
    off = torch.empty(N * K + 1, dtype=torch.bfloat16, device=DEV)[1:].view(N, K)
    off.copy_(w)
    for M in (1, 15, 17, 32):
        x = draw(M, K, seed=M)
        want, terms = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
        for splits in (0, 1):
            p = ragged._ext().gemm_parts(x, w, splits)
            assert p.dtype == torch.float32 and (not splits or p.shape[0] == 1)
            assert bool(((p.double().sum(0) - want).abs() <= 2.0 ** -20 * terms).all())
    if K % 256 == 0:
        p = ragged._ext().gemm_parts(x, off, 0)
        assert bool(((p.double().sum(0) - want).abs() <= 2.0 ** -20 * terms).all())
