"""Decode attention of batches whose contexts differ, in equal shares of their
tiles: contexts cut anywhere, whole ones, empty ones, windows, slopes, groups
wider than a tile and heads that don't divide the chip."""
import pytest
import torch

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]
DEV = "cuda"


def _want(q, kp, vp, table, lens, window, slopes):
    """Results and what the weights make of the values' absolutes, in 64 bits."""
    B, Hq, D = q.shape
    Hkv = kp.shape[1]
    out = torch.zeros(B, Hq, D, dtype=torch.float64, device=DEV)
    size = torch.zeros_like(out)
    for b, n in enumerate(lens):
        if n <= 0:
            continue
        pages = table[b].long()
        k = kp[pages].permute(1, 0, 2, 3).reshape(Hkv, -1, D)[:, :n].double()
        v = vp[pages].permute(1, 0, 3, 2).reshape(Hkv, -1, D)[:, :n].double()
        s = torch.matmul(q[b].view(Hkv, -1, D).double(),
                         k.transpose(1, 2).contiguous()) * D ** -0.5
        at = torch.arange(n, device=DEV)
        if slopes is not None:
            s = s + slopes.double().view(Hkv, -1, 1) * at
        if window > 0:
            s = s.masked_fill(at < n - window, float("-inf"))
        p = s.softmax(-1)
        out[b] = torch.matmul(p, v).view(Hq, D)
        size[b] = torch.matmul(p, v.abs()).view(Hq, D)
    return out, size


def _lens(kind, B, room, seed):
    g = torch.Generator().manual_seed(seed)
    if kind == "same":
        return [room // 2] * B
    lens = torch.randint(1, 200, (B,), generator=g).tolist()
    lens[0], lens[B // 2], lens[-1] = room, room - 1, 33
    if kind == "empty":
        lens[1] = lens[2] = lens[-1] = 0
    if kind == "first":
        lens = [room] + [1] * (B - 1)
    return lens


@pytest.mark.parametrize("B,Hkv,G,D,P,room,kind,window", [
    (33, 8, 4, 128, 32, 1600, "mixed", 0),
    (33, 8, 4, 128, 32, 1600, "empty", 0),
    (40, 8, 1, 128, 16, 1600, "first", 0),
    (33, 8, 4, 64, 8, 1600, "same", 0),
    (70, 8, 3, 32, 32, 1100, "mixed", 100),
    (33, 8, 8, 128, 32, 1600, "mixed", 0),
    (16, 8, 4, 128, 32, 6000, "empty", 0),
    (130, 1, 4, 128, 32, 1600, "mixed", 0),
    (52, 5, 4, 128, 32, 1600, "mixed", 777),
    (60, 1, 71, 64, 32, 1600, "mixed", 0),
    (9, 32, 1, 128, 32, 1600, "mixed", 0),
    (600, 1, 2, 64, 32, 1100, "empty", 0),
])
def test_shares(B, Hkv, G, D, P, room, kind, window):
    from bloombee_amd.ops import hip_ops
    lens = _lens(kind, B, room, B + D)
    Hq, maxp = Hkv * G, -(-room // P)
    assert hip_ops.decode_even(B, Hkv * -(-G // 16), maxp * P)
    gen = torch.Generator(device=DEV).manual_seed(B)
    rand = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(torch.bfloat16)
    np_ = sum(-(-max(n, 1) // P) for n in lens) + 1
    kp, vp = rand(np_, Hkv, P, D), rand(np_, Hkv, D, P)
    kp[0] = vp[0] = float("inf")                    # nobody's page
    order = (torch.randperm(np_ - 1, generator=gen, device=DEV) + 1).to(torch.int32)
    table = torch.zeros(B, maxp, dtype=torch.int32, device=DEV)
    at = 0
    for b, n in enumerate(lens):
        c = -(-n // P)
        table[b, :c] = order[at:at + c]
        at += c
        if n % P:                                   # behind the context
            kp[order[at - 1].long(), :, n % P:] = float("nan")
            vp[order[at - 1].long(), :, :, -(-(n % P) // 8) * 8:] = float("nan")
    q = rand(B, Hq, 1, D)
    slopes = torch.rand(Hq, generator=gen, device=DEV) * 0.01 if D == 32 else None
    ctx = torch.tensor(lens, dtype=torch.int32, device=DEV)
    run = lambda: hip_ops.attn_decode(q, kp, vp, table, ctx, D ** -0.5, window, -1, slopes)
    want, size = _want(q[:, :, 0], kp, vp, table, lens, window, slopes)
    # weights and results are rounded to eight binary places, by 2^-8 of them at most each;
    # scores of up to 2^4 are in 32 bits
    bound = lambda want, size: (size + want.abs()) * 1.01 * 2.0 ** -8 + 1e-5
    tol = bound(want, size)
    got = run()[:, :, 0].double()
    assert ((got - want).abs() <= tol).all(), ((got - want).abs() - tol).max()

    # captured, then other contexts
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run()
    for turn in range(3):
        lens = [max(0, n - 1 - turn * 31) if n else 0 for n in lens]
        ctx.copy_(torch.tensor(lens, dtype=torch.int32))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, run())
        want, size = _want(q[:, :, 0], kp, vp, table, lens, window, slopes)
        assert ((out[:, :, 0].double() - want).abs() <= bound(want, size)).all()


def test_which_batches():
    """Contexts with room for long ones that the chip has no even split of."""
    from bloombee_amd.ops import hip_ops
    even = hip_ops.decode_even
    assert not even(32, 8, 8192) and even(33, 8, 1536) and not even(33, 8, 1535)
    assert even(16, 8, 1536) and even(30, 8, 8192) and not even(15, 8, 8192)
    assert even(65, 8, 1024) and not even(65, 8, 1023)
    assert not even(65, 65, 4096) and not even(1025, 8, 4096)
    assert not even(1024, 8, 1 << 24)
