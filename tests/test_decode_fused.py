"""Decode GEMMs that take what follows them along, and the split of decode attention,
at the edges of their rules: rows up to which one launch does a GEMM, tiles of 16 and
32 columns, pieces of 128 columns of K shared out over eight or four waves."""
import pytest
import torch

from bloombee_amd import ops
from bloombee_amd.ops import reference as ref

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
ROWS = [1, 2, 4, 5, 16, 17, 25, 32]


def draw(*shape, seed=0, scale=1.0):
    gen = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=gen) * scale).bfloat16().to(DEV)


def close(got, want, scale=1.0):
    """Results are one bf16 rounding of 32-bit sums, 2^-9 of a value; another 2^-8 of
    the result's scale for hardware exponentials and reciprocals."""
    err = (got.double() - want).abs()
    assert bool((err <= 2.0 ** -8 * want.abs() + 2.0 ** -8 * scale).all()), err.max()


def rms(x, eps):
    x = x.double()
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("N,K", [(16, 128), (48, 256), (64, 1152), (80, 8064)])
def test_stream(M, N, K):
    x, w = draw(M, K, seed=1), draw(N, K, seed=2, scale=K ** -0.5)
    b, r = draw(N, seed=3), draw(M, N, seed=4)
    want = x.double() @ w.double().T
    close(ops.hip_ops.gemm_stream(x, w, None, None, -1.0), want)
    close(ops.hip_ops.gemm_stream(x, w, r, b, -1.0), want + b.double() + r.double())
    close(ops.hip_ops.gemm_stream(x, w, r, None, 1e-5),
          rms(x, 1e-5) @ w.double().T + r.double())


# (columns, K, parts of K up to 4 rows and up to 8): ends of the rule; a wave's pieces
# fewer than four, four and more, some waves without any
@pytest.mark.parametrize("M", [1, 3, 4, 5, 7, 8, 9])
@pytest.mark.parametrize("N,K,few,more", [
    (16, 1024, 0, 0), (16, 1152, 2, 2), (1024, 2048, 2, 2), (1024, 2176, 4, 2),
    (1040, 3072, 2, 2), (2048, 1152, 2, 2), (2064, 2048, 0, 0), (32, 4096, 4, 2),
    (48, 4224, 4, 2)])
def test_stream_in_parts(M, N, K, few, more):
    x, w = draw(M, K, seed=1), draw(N, K, seed=2, scale=K ** -0.5)
    b, r = draw(N, seed=3), draw(M, N, seed=4)
    assert ops.hip_ops.stream_parts(M, N, K) == (few if M <= 4 else more if M <= 8
                                                 else 0)
    want = x.double() @ w.double().T
    close(ops.hip_ops.gemm_stream(x, w, None, None, -1.0), want)
    close(ops.hip_ops.gemm_stream(x, w, r, b, -1.0), want + b.double() + r.double())
    # what is not finite stays in its row of x or of w
    x[M - 1, K - 1], w[5, 0] = float("inf"), float("nan")
    got, want = ops.hip_ops.gemm_stream(x, w, None, None, -1.0), x.float() @ w.float().T
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isinf(), want.isinf())


def test_stream_refuses_what_it_cannot_do():
    for M, N, K in ((33, 16, 128), (1, 24, 128), (1, 16, 192)):
        with pytest.raises(RuntimeError):
            ops.hip_ops.gemm_stream(draw(M, K), draw(N, K), None, None, -1.0)


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("I,K", [(32, 256), (96, 768), (1024, 512)])
def test_gated_product(M, I, K):
    x, w = draw(M, K, seed=1), draw(2 * I, K, seed=2, scale=K ** -0.5)
    z = rms(x, 1e-5) @ w.double().T
    want = torch.nn.functional.silu(z[:, :I]) * z[:, I:]
    assert ops.fuse_norm_linear_ok(x, w)
    close(ops.linear_swiglu(x, w, 1e-5), want)


@pytest.mark.parametrize("M", [17, 32])
def test_large_weights_keep_the_split_gemm(M):
    """Beyond 16 rows and 2^25 weights: the split forms, with the rows' squares."""
    K = 4096
    x = draw(M, K, seed=1)
    w = draw(8256, K, seed=2, scale=K ** -0.5)
    assert not ops.streams_weights(x, w) and ops.streams_weights(x[:16], w)
    assert ops.streams_weights(x, w[:8192])
    z = rms(x, 1e-5) @ w.double().T
    want = torch.nn.functional.silu(z[:, :4128]) * z[:, 4128:]
    close(ops.linear_swiglu(x, w, 1e-5), want)
    kp, vp = draw(4, 43, 16, 64, seed=4), draw(4, 43, 64, 16, seed=5)
    table = torch.arange(4, device=DEV, dtype=torch.int32).view(1, 4)
    start = torch.tensor([9], dtype=torch.int32, device=DEV)
    cos, sin = (t.to(DEV) for t in ops.rope_cos_sin(64, 128))
    z = z.view(1, M, -1).float().cpu()
    kw, vw = kp.float().cpu(), vp.float().cpu()
    ops.rope_kv_write_(z, 43, 43, cos.cpu(), sin.cpu(), None, kw, vw, table.cpu(),
                       start.cpu())
    got = ops.linear_rope_kv(x[None], w, 1e-5, 43, 43, cos, sin, None, kp, vp, table,
                             start)
    close(got[..., :43 * 64].cpu(), z[..., :43 * 64].double())
    close(kp.cpu(), kw.double())
    close(vp.cpu(), vw.double())


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("Hq,Hkv,D,P,K", [(4, 2, 64, 16, 256), (2, 1, 128, 8, 512),
                                          (8, 2, 32, 16, 1024)])
@pytest.mark.parametrize("ids", [False, True])
def test_rotations_and_pages(M, Hq, Hkv, D, P, K, ids):
    B = 1 if M % 2 else 2
    T = M // B
    x = draw(B, T, K, seed=1)
    w = draw((Hq + 2 * Hkv) * D, K, seed=2, scale=K ** -0.5)
    start = torch.tensor([5, 2 * P - 1][:B], dtype=torch.int32, device=DEV)
    room = int(start.max()) + T
    maxp = -(-room // P) + 1
    table = torch.randperm(B * maxp, generator=torch.Generator().manual_seed(3))
    table = table.view(B, maxp).int().to(DEV)
    kp, vp = draw(B * maxp, Hkv, P, D, seed=4), draw(B * maxp, Hkv, D, P, seed=5)
    cos, sin = (t.to(DEV) for t in ops.rope_cos_sin(D, 128))
    pos = None
    if ids:
        pos = torch.arange(M, device=DEV, dtype=torch.int32).view(B, T) % 7 + 3
    # the same in steps: plain projection, then the CPU form of the pages' writer
    z = (rms(x, 1e-5) @ w.double().T).float().cpu()
    kw, vw = kp.float().cpu(), vp.float().cpu()
    ops.rope_kv_write_(z, Hq, Hkv, cos.cpu(), sin.cpu(),
                       pos.cpu() if ids else None, kw, vw, table.cpu(), start.cpu())
    got = ops.linear_rope_kv(x, w, 1e-5, Hq, Hkv, cos, sin, pos, kp, vp, table,
                             start)
    close(got[..., :Hq * D].cpu(), z[..., :Hq * D].double())
    close(kp.cpu(), kw.double())
    close(vp.cpu(), vw.double())


def test_head_norms_ride_the_rotation():
    B, T, Hq, Hkv, D, P = 2, 3, 4, 2, 128, 16
    z = draw(B, T, (Hq + 2 * Hkv) * D, seed=1)
    qw, kw = draw(D, seed=2) + 1, draw(D, seed=3) + 1
    table = torch.arange(4, dtype=torch.int32, device=DEV).view(B, 2)
    start = torch.tensor([0, 15], dtype=torch.int32, device=DEV)
    cos, sin = (t.to(DEV) for t in ops.rope_cos_sin(D, 64))
    pages = [torch.zeros(4, Hkv, *s, dtype=torch.bfloat16, device=DEV)
             for s in ((P, D), (D, P))]
    want = z.float().cpu()
    wp = [p.float().cpu() for p in pages]
    norms = (qw, kw, 1e-6)
    ops.rope_kv_write_(want, Hq, Hkv, cos.cpu(), sin.cpu(), None, *wp, table.cpu(),
                       start.cpu(), head_norms=(qw.float().cpu(), kw.float().cpu(),
                                                1e-6))
    ops.rope_kv_write_(z, Hq, Hkv, cos, sin, None, *pages, table, start,
                       head_norms=norms)
    close(z[..., :Hq * D].cpu(), want[..., :Hq * D].double(), 4.0)
    for p, q in zip(pages, wp):
        close(p.cpu(), q.double(), 4.0)


@pytest.mark.parametrize("B,T", [(1, 63), (1, 64), (64, 1), (3, 23), (2, 100), (9, 8)])
@pytest.mark.parametrize("Hq,Hkv,D,P", [(4, 2, 128, 16), (3, 1, 64, 8), (2, 1, 32, 32),
                                        (2, 2, 256, 16)])
@pytest.mark.parametrize("norms", [False, True])
def test_octets_of_tokens(B, T, Hq, Hkv, D, P, norms):
    """Many tokens: octets that begin or end within a sequence, one token each; the
    slots around them stay as they are."""
    qkv = draw(B, T, (Hq + 2 * Hkv) * D, seed=1)
    start = (torch.arange(B, dtype=torch.int32) * 5 + 3).to(DEV)
    maxp = -(-(int(start.max()) + T) // P)
    gen = torch.Generator().manual_seed(3)
    table = torch.randperm(B * maxp, generator=gen).view(B, maxp).int().to(DEV)
    kp, vp = draw(B * maxp, Hkv, P, D, seed=4), draw(B * maxp, Hkv, D, P, seed=5)
    cos, sin = (t.to(DEV) for t in ops.rope_cos_sin(D, 256))
    pos = (torch.arange(B * T, dtype=torch.int32, device=DEV).view(B, T) % 200
           if T % 2 else None)
    hn = (draw(D, seed=6) + 1, draw(D, seed=7) + 1, 1e-6) if norms else None
    want, kw, vw = qkv.float().cpu(), kp.float().cpu(), vp.float().cpu()
    ops.rope_kv_write_(want, Hq, Hkv, cos.cpu(), sin.cpu(),
                       None if pos is None else pos.cpu(), kw, vw, table.cpu(),
                       start.cpu(), head_norms=hn and (hn[0].float().cpu(),
                                                       hn[1].float().cpu(), 1e-6))
    ops.rope_kv_write_(qkv, Hq, Hkv, cos, sin, pos, kp, vp, table, start, head_norms=hn)
    scale = 4.0 if norms else 1.0
    close(qkv[..., :Hq * D].cpu(), want[..., :Hq * D].double(), scale)
    close(kp.cpu(), kw.double(), scale)
    assert torch.equal(vp.cpu().float(), vw)


@pytest.mark.parametrize("B,Hq,Hkv,D,room,lengths", [
    (1, 4, 1, 128, 128, [1]),                 # one split, one token
    (1, 4, 2, 128, 300, [300]),               # two splits
    (2, 8, 2, 128, 4096, [5, 4096]),          # a short context in a wide table
    (1, 71, 1, 64, 2000, [777]),              # a group in five chunks
    (65, 8, 8, 64, 2100, None),               # more units than fit: even shares
    (3, 16, 8, 128, 264, [264, 1, 257]),      # eight waves: one split
    (3, 8, 8, 64, 336, [330, 31, 256]),
    (16, 32, 8, 128, 480, None),              # a split of two that is not there
    (2, 16, 8, 128, 4000, [4000, 511]),       # one of many
    (32, 8, 8, 32, 240, None), (32, 32, 8, 64, 1000, None),
    (24, 8, 8, 128, 600, None), (17, 8, 8, 128, 600, None),   # two tiles and more a wave
])
@pytest.mark.parametrize("P", [8, 16, 24])        # 24: pages found by division
def test_decode_attention_splits(B, Hq, Hkv, D, room, lengths, P):
    gen = torch.Generator().manual_seed(B)
    if lengths is None:
        lengths = torch.randint(1, room + 1, (B,), generator=gen).tolist()
    maxp = -(-room // P)
    kp, vp = draw(B * maxp, Hkv, P, D, seed=1), draw(B * maxp, Hkv, D, P, seed=2)
    table = torch.randperm(B * maxp, generator=gen).view(B, maxp).int().to(DEV)
    qkv = draw(B, 1, (Hq + 2 * Hkv) * D, seed=3)
    start = torch.tensor([n - 1 for n in lengths], dtype=torch.int32, device=DEV)
    q = qkv[..., :Hq * D].view(B, 1, Hq, D).transpose(1, 2)
    want = ref.attn_paged(q.float(), kp.float(), vp.float(), table, start.long())
    got = ops.attn_paged_qkv(qkv, Hq, Hkv, kp, vp, table, start)
    # weights enter the value product in bf16: 2^-9 of the largest value
    err = (got.view(B, Hq, D).float() - want[:, :, 0]).abs().max()
    assert err <= 2 * 4.5 * 2.0 ** -9, err


def off(t):
    """The same at two bytes into a line."""
    wide = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)
    wide[1:].copy_(t.reshape(-1))
    assert wide[1:].data_ptr() % 16 == 2
    return wide[1:].view(t.shape)


@pytest.mark.parametrize("M", [1, 5, 16, 17, 32])
def test_rows_at_any_address(M):
    x, w, r = draw(M, 512, seed=1), draw(64, 512, seed=2, scale=0.05), draw(M, 64)
    assert torch.equal(ops.linear(off(x), w, residual=r), ops.linear(x, w, residual=r))
    assert torch.equal(ops.linear(x, off(w)), ops.linear(x, w))
    assert torch.equal(ops.linear_swiglu(off(x), w, 1e-5), ops.linear_swiglu(x, w, 1e-5))
    table = torch.arange(4, device=DEV, dtype=torch.int32).view(1, 4)
    start = torch.tensor([9], dtype=torch.int32, device=DEV)
    cos, sin = (t.to(DEV) for t in ops.rope_cos_sin(32, 128))
    w = draw(128, 512, seed=2, scale=0.05)
    outs = []
    for rows in (x, off(x)):
        kp, vp = (torch.zeros(4, 1, *s, dtype=torch.bfloat16, device=DEV)
                  for s in ((16, 32), (32, 16)))
        q = ops.linear_rope_kv(rows[None], w, 1e-5, 2, 1, cos, sin, None, kp, vp, table,
                               start)
        outs.append((q[..., :64], kp, vp))
    for a, b in zip(*outs):
        assert torch.equal(a, b)


def test_no_rows():
    x, w = draw(0, 512), draw(64, 512)
    for rows in (x, x.view(0, 1, 512), x.view(1, 0, 512)):
        assert ops.linear(rows, w).shape == (*rows.shape[:-1], 64)
        assert ops.linear_swiglu(rows, w, 1e-5).shape == (*rows.shape[:-1], 32)


@pytest.mark.parametrize("N,K", [(512, 14336), (4096, 512), (4096, 14336), (4160, 512),
                                 (4160, 1024), (4608, 4096), (8192, 4096), (8256, 3072),
                                 (12288, 1024), (16384, 1024), (18176, 2048),
                                 (32000, 1024)])
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32])
def test_products_on_both_sides_of_their_rules(M, N, K):
    """Rounds of workgroups full and nearly empty: whatever kernel takes a product, its
    result is one rounding of a 32-bit sum."""
    x, w, r = draw(M, K, seed=1), draw(N, K, seed=2, scale=K ** -0.5), draw(M, N, seed=3)
    z = x.double() @ w.double().T
    close(ops.linear(x, w), z)
    close(ops.linear(x, w, residual=r), z + r.double())
    n = rms(x, 1e-5) @ w.double().T
    want = torch.nn.functional.silu(n[:, :N // 2]) * n[:, N // 2:]
    close(ops.linear_swiglu(x, w, 1e-5), want)
    if N % 192 == 0 or N == 8192:            # heads of 64, as many of each kind
        H = N // 64
        Hkv = 1 if N == 8192 else H // 3
        Hq = H - 2 * Hkv
        kp, vp = (torch.zeros(4, Hkv, *s, dtype=torch.bfloat16, device=DEV)
                  for s in ((16, 64), (64, 16)))
        table = torch.arange(4, device=DEV, dtype=torch.int32).view(1, 4)
        start = torch.tensor([9], dtype=torch.int32, device=DEV)
        cos, sin = (t.to(DEV) for t in ops.rope_cos_sin(64, 128))
        n = n.view(1, M, -1).float().cpu()
        kw, vw = kp.float().cpu(), vp.float().cpu()
        ops.rope_kv_write_(n, Hq, Hkv, cos.cpu(), sin.cpu(), None, kw, vw, table.cpu(),
                           start.cpu())
        got = ops.linear_rope_kv(x[None], w, 1e-5, Hq, Hkv, cos, sin, None, kp, vp, table,
                                 start)
        close(got[..., :Hq * 64].cpu(), n[..., :Hq * 64].double())
        close(kp.cpu(), kw.double())
        close(vp.cpu(), vw.double())


def test_rules_of_decode_products():
    """Both sides of each rule are reached by the sizes above."""
    sums, glu, rope = (getattr(ops.hip_ops, "stream_" + n)
                       for n in ("sums", "swiglu", "rope"))
    assert sums(1, 4096, 14336) and not sums(32, 4096, 14336)
    assert not sums(1, 4160, 512) and sums(1, 4160, 1024)
    assert sums(16, 4608, 4096) and not sums(1, 4608, 6400)
    assert sums(8, 9216, 4096) and not sums(9, 9216, 4096)
    assert sums(16, 18176, 2048) and not sums(1, 32000, 1024)
    assert sums(32, 8192, 4096) and not sums(32, 8256, 3072)
    assert glu(32, 8192, 4096) and glu(4, 16384, 1024) and not glu(5, 16384, 1024)
    assert glu(32, 18176, 2048) and not glu(16, 32000, 1024) and not glu(1, 18176, 512)
    assert rope(17, 12288, 1024) and not rope(16, 4608, 4096)
    assert rope(17, 8192, 4096) and not rope(17, 18176, 2048)


@pytest.mark.parametrize("B,Hq,Hkv,D,room,window", [
    (1, 4, 2, 128, 4096, 300),                # splits ahead of the window
    (2, 8, 4, 256, 4096, 1024),
    (1, 8, 2, 64, 4096, 1),
    (1, 8, 4, 512, 300, 0),                   # splits of 32 tokens
    (2, 4, 1, 512, 4096, 700),
    (3, 16, 1, 512, 96, 0),
])
def test_decode_attention_without_some_splits(B, Hq, Hkv, D, room, window):
    """Splits ahead of a window or beyond a short context in a wide table hold nothing."""
    lengths = [room, 33, 1][:B]
    maxp = -(-room // 16)
    kp, vp = draw(B * maxp, Hkv, 16, D, seed=1), draw(B * maxp, Hkv, D, 16, seed=2)
    gen = torch.Generator().manual_seed(B)
    table = torch.randperm(B * maxp, generator=gen).view(B, maxp).int().to(DEV)
    q = draw(B, Hq, 1, D, seed=3)
    start = torch.tensor([n - 1 for n in lengths], device=DEV)
    want = ref.attn_paged(q.float(), kp.float(), vp.float(), table, start,
                          sliding_window=window or None)
    got = ops.attn_paged(q, kp, vp, table, start, window=window)
    # weights enter the value product in bf16, 2^-9 of the largest value; so does the
    # result
    err = (got.float() - want).abs().max()
    assert err <= 2 * 4.5 * 2.0 ** -9, err
