"""Routing ahead of the experts and their sum behind them, at the edges: one expert,
64, all of them chosen, equal and missing logits, rows of either path (two weight
streams up to 32 rows, sorted tiles beyond)."""
import pytest
import torch

from bloombee_amd import ops
from bloombee_amd.ops import ragged

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def draw(*shape, seed=0, scale=1.0):
    gen = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=gen) * scale).bfloat16().to(DEV)


def rms(x, w, eps):
    x = x.double()
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w.double()


@pytest.mark.parametrize("N,H,E,top", [(1, 8, 1, 1), (5, 264, 8, 2), (33, 4096, 8, 8),
                                       (3, 2048, 64, 6), (2, 16384, 5, 3)])
def test_norm_and_routing(N, H, E, top):
    a, r = draw(N, H, seed=1), draw(N, H, seed=2)
    w, router = draw(H, seed=3, scale=0.1) + 1, draw(E, H, seed=4, scale=H ** -0.5)
    h, y, ids, wts = ops.hip_ops.norm_route(a, r, w, router, top, 1e-5)
    assert torch.equal(h, a + r)
    want = rms(h, w, 1e-5)
    # one rounding to bf16
    assert bool(((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-6).all())
    # from its own norm on: logits are bf16 results of 32-bit sums
    logits = y.double() @ router.double().T
    got = logits.gather(1, ids.long())
    step = 2.0 ** -8 * logits.abs().amax(1, keepdim=True) + 1e-6
    kth = logits.topk(top, -1).values
    assert bool(((got - kth).abs() <= 2 * step).all())
    assert all(len(set(row)) == top for row in ids.tolist())
    soft = torch.softmax(got, -1)
    # the weights are bf16 themselves
    assert bool(((wts.double() - soft).abs() <= 4 * step + 2.0 ** -9).all())


def test_equal_and_missing_logits_choose_distinct_experts():
    a = draw(3, 64, seed=1)
    router = draw(6, 64, seed=2)
    router[2] = router[4]
    a[1] = 0.0                               # all equal
    a[2, 5] = float("nan")                   # none there
    _, y, ids, wts = ops.hip_ops.norm_route(a, None, None, router, 3, 0.0)
    assert y.data_ptr() == a.data_ptr()
    assert all(len(set(row)) == 3 and 0 <= min(row) and max(row) < 6
               for row in ids.tolist())
    assert ids[1].tolist() == [0, 1, 2]      # the first of equal ones
    assert bool(((wts[:2].sum(1) - 1).abs() <= 3 * 2.0 ** -10).all())
    assert bool(wts[2].isnan().all())


@pytest.mark.parametrize("N", [1, 31, 32, 33, 200])
@pytest.mark.parametrize("E,top,H,I", [(4, 2, 256, 320), (1, 1, 64, 64),
                                       (8, 3, 192, 128)])
def test_routed_mlp(N, E, top, H, I):
    a, r = draw(N, H, seed=1), draw(N, H, seed=2)
    w, router = draw(H, seed=3, scale=0.1) + 1, draw(E, H, seed=4)
    up = draw(E, 2 * I, H, seed=5, scale=H ** -0.5)
    down = draw(E, H, I, seed=6, scale=I ** -0.5)
    assert ops.routed_mlp_ok(a, up, down, top)
    h, y, ids, wts = ops.hip_ops.norm_route(a, r, w, router, top, 1e-5)
    want = torch.zeros(N, H, dtype=torch.float64, device=DEV)
    tol = torch.zeros_like(want)
    for n in range(N):
        for c in range(top):
            e, wt = int(ids[n, c]), float(wts[n, c])
            g, u = (y[n].double() @ up[e].double().T).chunk(2)
            act = torch.nn.functional.silu(g) * u
            row = wt * (act @ down[e].double().T)
            want[n] += row
            # an expert's row and the sums over them are bf16, 2^-9 of them; so
            # are gate, up and activation, whose roundings add up like random
            # ones (five deviations, three roundings)
            tol[n] += 2.0 ** -9 * ((1 + top) * row.abs() + 15 * wt * (
                act.square() @ down[e].double().square().T).sqrt())
    got = ops.routed_mlp(y, router, up, down, top)
    # hardware exponentials stay far below
    assert bool(((got.double() - want).abs()
                 <= tol + 2.0 ** -8 * want.abs() + 1e-6).all())
    got = ops.routed_mlp(a, router, up, down, top, r, (w, 1e-5))
    want = want + h.double()
    assert bool(((got.double() - want).abs()
                 <= tol + 2.0 ** -8 * want.abs() + 1e-6).all())


@pytest.mark.parametrize("counts,K,F,W", [
    ([40, 0, 1, 64, 65], 64, 64, 320),               # tiles of 64 rows, two steps each
    ([129, 1, 300, 0, 127], 192, 192, 64),           # tiles of 128
    ([0, 1030, 128, 2, 2400], 128, 320, 64),         # groups of 5 and 4, of 7, 6 and 6
    # tiles of every height, with fewer steps than buffers and more, columns that end
    # within a tile
    ([57, 97, 38], 320, 192, 320),                   # 96 rows
    ([87, 1, 200], 448, 320, 192),                   # 128
    ([118, 161, 75], 64, 64, 64),                    # 160
    ([148, 193, 103], 128, 448, 320),                # 192
    ([179, 257, 101], 448, 128, 448),                # 101 to 179 rows, half as wide
    ([193, 385, 300, 513], 320, 448, 64),            # 97 to 193
    ([513, 770, 1], 64, 320, 320),
    # 40 tiles or more, 256 columns wide: 97, 128, 150, 171, 192, 200 and 256 rows
    ([193, 256, 300, 342, 384, 400, 512] * 4, 192, 832, 1600),
    ([400, 130] * 12, 128, 896, 1600),
])
@pytest.mark.parametrize("planes", [1, 2])
def test_order_of_tiles(counts, K, F, W, planes):
    """Experts of none to many row tiles, columns that end within a tile."""
    E, N = len(counts), sum(counts)
    gen = torch.Generator().manual_seed(1)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    ids = ids[torch.randperm(N, generator=gen)].to(DEV)
    wts = torch.rand(N, generator=gen).to(DEV) + 0.5
    h = draw(N, K, seed=2)
    up = draw(E, planes, F, K, seed=3, scale=K ** -0.5)
    down = draw(E, W, F, seed=4, scale=F ** -0.5)
    rt = ragged.Routing(ids.int()[:, None], wts[:, None], None)
    got = ragged.moe_experts(h, up, down, rt)[:, 0]
    for e in range(E):
        at = ids == e
        z = torch.einsum("nk,pfk->pnf", h[at].double(), up[e].double())
        act = (torch.nn.functional.silu(z[0]) * z[1] if planes == 2
               else z[0].clamp(min=0) ** 2)
        w = wts[at].double()[:, None]
        want = act @ down[e].double().T * w
        # the result's rounding, 2^-9, and that of activations, whose exponentials
        # and reciprocals take as much again
        tol = 2.0 ** -8 * want.abs() + 2.0 ** -8 * w * (act.abs()
                                                      @ down[e].double().abs().T)
        assert bool(((got[at].double() - want).abs() <= tol + 1e-6).all())


@pytest.mark.parametrize("N", [3, 40])
def test_rows_at_any_address(N):
    """Views that begin at two bytes into a line: rows are copied, weights are left to
    the loop over the experts."""
    E, top, H, I = 4, 2, 128, 64
    a, router = draw(N, H, seed=1), draw(E, H, seed=4)
    up = draw(E, 2 * I, H, seed=5, scale=H ** -0.5)
    down = draw(E, H, I, seed=6, scale=I ** -0.5)

    def off(t):
        wide = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)
        wide[1:].copy_(t.reshape(-1))
        return wide[1:].view(t.shape)

    assert torch.equal(ops.routed_mlp(off(a), router, up, down, top),
                       ops.routed_mlp(a, router, up, down, top))
    assert ops.routed_mlp_ok(off(a), up, down, top)
    assert not ops.routed_mlp_ok(a, off(up), down, top)
    assert not ops.routed_mlp_ok(a, up, off(down), top)


@pytest.mark.parametrize("bits", [0x7fc0, 0xffc0 - 0x10000], ids=["nan", "-nan"])
def test_order_of_unusual_logits(bits):
    """NaN of either sign above all numbers, both zeros equal, infinities in place."""
    a = torch.zeros(1, 64, dtype=torch.bfloat16, device=DEV)
    a[0, 0] = 1.0
    router = torch.zeros(6, 64, dtype=torch.bfloat16, device=DEV)
    router[:, 0] = torch.tensor([1.0, float("inf"), -float("inf"), 3.0, 0.0, 2.0])
    router.view(torch.int16)[4, 0] = bits
    _, _, ids, wts = ops.hip_ops.norm_route(a, None, None, router, 5, 0.0)
    assert ids[0].tolist() == [4, 1, 3, 5, 0]
    assert bool(wts.isnan().all())
    # products that vanish in bf16 keep their sign
    a[0, 0] = 2.0 ** -100
    router[:, 0] = torch.tensor([-2.0 ** -40, 2.0 ** -40, -1.0, 0.0, -1.0, -1.0])
    _, _, ids, wts = ops.hip_ops.norm_route(a, None, None, router, 5, 0.0)
    assert ids[0].tolist() == [0, 1, 3, 2, 4]
    assert bool(((wts - 0.2).abs() <= 2.0 ** -10).all())


@pytest.mark.parametrize("flat", [False, True])
def test_more_rows_than_32_bits_of_bytes_reach(flat):
    """Batches of 2^32 bytes are taken in parts, weights laid out (N, top) or not."""
    N, K, top = 1 << 15, 1 << 16, 2
    h = torch.zeros(N, K, dtype=torch.bfloat16, device=DEV)
    at = torch.tensor([0, 1, N // 2 - 1, N // 2, N - 2, N - 1], device=DEV)
    h[at] = draw(len(at), K, seed=1)
    up = draw(2, 1, 64, K, seed=2, scale=K ** -0.5)
    down = draw(2, 64, 64, seed=3, scale=0.125)
    gen = torch.Generator().manual_seed(4)
    ids = torch.rand(N, 2, generator=gen).argsort(1).int().to(DEV)
    wts = torch.rand(N, top, generator=gen).to(DEV)
    got = ragged._ext().moe_experts(h, up, down, ids, wts.flatten() if flat else wts,
                                    False, 0.0, 1.0, 0.0, False)
    x, e = h[at].double(), ids[at].long()
    act = torch.relu(torch.einsum("nk,etk->net", x, up[:, 0].double())).square()
    act = act[torch.arange(len(at), device=DEV)[:, None], e]         # (n, top, 64)
    back = down.double()[e]                                          # (n, top, 64, 64)
    w = wts[at].double()[..., None]
    want = w * (back * act[:, :, None]).sum(-1)
    # an activation and its row are rounded to 16 bits, 2^-9 of each
    tol = 2.0 ** -8 * (want.abs() + w * (back.abs() * act[:, :, None]).sum(-1))
    assert bool(((got[at].double() - want).abs() <= tol + 1e-6).all())
    zero = torch.ones(N, dtype=torch.bool, device=DEV)
    zero[at] = False
    assert not got[zero].any()


@pytest.mark.parametrize("N,E,top,planes,K,F,Wp", [
    (1, 4, 2, 2, 64, 64, 64),                # one row, one stage of K
    (32, 1, 1, 2, 192, 192, 320),            # all rows of one expert
    (17, 2, 1, 1, 320, 192, 4160),           # a tile's last columns
    (16, 8, 2, 2, 128, 4096, 8192),          # enough columns for wide tiles
    (9, 64, 6, 1, 576, 1088, 64), (31, 300, 3, 2, 64, 128, 192)])
@pytest.mark.parametrize("win", [False, True])
def test_few_tokens(N, E, top, planes, K, F, Wp, win):
    h = draw(N, K, seed=1)
    up = draw(E, planes, F, K, seed=2, scale=K ** -0.5)
    down = draw(E, Wp, F, seed=3, scale=F ** -0.5)
    gen = torch.Generator().manual_seed(4)
    ids = torch.rand(N, E, generator=gen).argsort(1)[:, :top].int()
    wts = torch.rand(N, top, generator=gen) + 0.5
    skipped = torch.rand(N, top, generator=gen) < 0.2
    got = ragged._ext().moe_experts(h, up, down, ids.masked_fill(skipped, -1).to(DEV),
                                    wts.to(DEV), win, float("inf"), 1.0, 0.0, False)
    x, up, down = (t.double().cpu() for t in (h, up, down))
    for n in range(N):
        for c in range(top):
            if skipped[n, c]:
                continue
            e, w = int(ids[n, c]), float(wts[n, c])
            z = up[e] @ x[n] * (w if win else 1.0)
            act = (torch.nn.functional.silu(z[0]) * z[1] if planes == 2 else
                   torch.relu(z[0]).square())
            want = down[e] @ act * (1.0 if win else w)
            # an activation and its row are rounded to 16 bits, 2^-9 of each
            tol = 2.0 ** -8 * (want.abs() + (1.0 if win else w)
                               * (down[e].abs() @ act.abs()))
            assert bool(((got[n, c].double().cpu() - want).abs() <= tol + 1e-6).all())
