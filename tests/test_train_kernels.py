"""Fused steps of the training path against their plain forms: both are compared with
the plain form in 64 bits, and the fused one may be no further away."""
import pytest
import torch

from bloombee_amd import ops
from bloombee_amd.ops import training

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def draw(*shape, seed=0, scale=1.0):
    gen = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=gen) * scale).to(torch.bfloat16).to(DEV)


def away(x, exact):
    return float((x.double() - exact).norm() / exact.norm().clamp_min(1e-30))


def check(fused, plain, exact):
    """Both round their results to bf16; a tenth more covers another order of
    rounding, 1e-6 results that are exact."""
    for f, p, e in zip(fused, plain, exact):
        assert f.shape == p.shape and f.dtype == p.dtype
        assert away(f, e) <= 1.1 * away(p, e) + 1e-6, (away(f, e), away(p, e))


def grads(f, xs, gs, dtype=None):
    xs = [x.detach().to(dtype or x.dtype).requires_grad_(True) for x in xs]
    out = f(*xs)
    out = out if isinstance(out, tuple) else (out,)
    return [*out, *torch.autograd.grad(out, xs, [g.to(o.dtype) for g, o
                                                 in zip(gs, out)])]


def attention(Hq, Hkv, D, T, start):
    cos, sin = ops.rope_cos_sin(D, start + T + 3)
    cos, sin = cos.to(DEV), sin.to(DEV)
    scale = D ** -0.5
    fused = lambda x: training.rope_attention(x, cos, sin, Hq, Hkv, start, scale)
    plain = lambda x: training._attention(x, cos, sin, Hq, Hkv, start, scale)

    def exact(x):
        B, X = x.shape[0], Hq + 2 * Hkv
        q, k, v = x.view(B, T, X, D).split([Hq, Hkv, Hkv], 2)
        c, s = (t[start:start + T, None].double() for t in (cos, sin))

        def rot(t):
            a, b = t.chunk(2, -1)
            return torch.cat([a * c - b * s, b * c + a * s], -1)

        q, k = rot(q), rot(k).repeat_interleave(Hq // Hkv, 2)
        v = v.repeat_interleave(Hq // Hkv, 2)
        sc = torch.einsum("bthd,bshd->bhts", q, k) * scale
        i = torch.arange(T, device=DEV)
        p = torch.softmax(sc.masked_fill(i > i[:, None], float("-inf")), -1)
        return torch.einsum("bhts,bshd->bthd", p, v).reshape(B, T, Hq * D)

    return fused, plain, exact


@pytest.mark.parametrize("case", [
    # B, Hq, Hkv, D, T, start: rows (token, head of the group) go in tiles of 128
    # and 64, keys in tiles of 64 and 32
    (1, 4, 4, 128, 1, 0), (1, 4, 1, 128, 2, 0), (2, 8, 2, 128, 31, 5),
    (1, 8, 2, 128, 32, 0), (3, 8, 2, 128, 33, 0), (1, 2, 2, 64, 63, 0),
    (2, 6, 2, 64, 64, 7), (1, 4, 2, 128, 65, 0), (1, 4, 4, 64, 128, 0),
    (1, 4, 4, 128, 129, 1), (2, 12, 4, 128, 200, 0), (1, 32, 8, 128, 515, 0),
], ids=lambda c: "-".join(map(str, c)))
def test_attention(case):
    B, Hq, Hkv, D, T, start = case
    x = draw(B, T, (Hq + 2 * Hkv) * D, seed=T)
    g = draw(B, T, Hq * D, seed=T + 1)
    fused, plain, exact = attention(Hq, Hkv, D, T, start)
    assert training._fused(x)
    check(grads(fused, [x], [g]), grads(plain, [x], [g]),
          grads(exact, [x], [g], torch.float64))
    with torch.no_grad():
        assert torch.equal(fused(x), fused(x.clone().requires_grad_(True)))


@pytest.mark.parametrize("case", [
    # tiles of 64 rows on their way three ahead, heads that divide 64 and others: less
    # than the ring holds, its size, more; waves that join late and leave early
    (1, 6, 2, 128, 150, 0), (1, 14, 2, 64, 100, 3), (1, 64, 1, 64, 9, 0),
    (1, 71, 1, 128, 40, 0), (1, 128, 1, 64, 70, 0), (2, 4, 4, 128, 191, 0),
    (1, 4, 4, 64, 193, 0), (1, 8, 4, 128, 257, 0), (1, 10, 2, 128, 97, 0),
], ids=lambda c: "-".join(map(str, c)))
def test_gradients_of_keys_and_values(case):
    """Every head, also where a row's gradient or log-sum is not a number: keys it does not
    see, of other tiles than its own, keep what they have."""
    B, Hq, Hkv, D, T, start = case
    x = draw(B, T, (Hq + 2 * Hkv) * D, seed=T)
    g = draw(B, T, Hq * D, seed=T + 1)
    fused, plain, exact = attention(Hq, Hkv, D, T, start)
    want = grads(fused, [x], [g])
    check(want, grads(plain, [x], [g]), grads(exact, [x], [g], torch.float64))
    g[0, 0, 0] = float("nan")                 # the first token sees the first key alone
    got = grads(fused, [x], [g])[1].view(B, T, Hq + 2 * Hkv, D)
    want = want[1].view(B, T, Hq + 2 * Hkv, D)
    assert bool(got[0, 0].isnan().any())
    assert torch.equal(got[0, 64:], want[0, 64:]) and torch.equal(got[1:], want[1:])


@pytest.mark.parametrize("shape", [(1, 8), (3, 5, 256), (7, 2056), (2, 3, 4096),
                                   (5, 16384)], ids=str)
def test_norms(shape):
    x, a = draw(*shape, seed=1), draw(*shape, seed=2)
    w = draw(shape[-1], seed=3, scale=0.2) + 1
    gh, gy = draw(*shape, seed=4), draw(*shape, seed=5)

    def add_norm(f):
        return lambda a, x: f(a, x, w, 1e-5)

    def plain(a, x):
        h = x + a
        return h, training._rms(h, w, 1e-5)

    def exact(a, x):
        h = (x + a)
        h = h + (h.bfloat16().double() - h).detach()   # the sum is a bf16 result
        return h, h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + 1e-5) * w.double()

    check(grads(add_norm(training.add_norm), [a, x], [gh, gy]),
          grads(plain, [a, x], [gh, gy]), grads(exact, [a, x], [gh, gy], torch.float64))
    one = grads(lambda t: training.norm(t, w, 1e-5), [x], [gh, gy])
    two = grads(lambda t: training.add_norm(torch.zeros_like(t), t, w, 1e-5), [x],
                [gh, gy])
    for u, v in zip(one, two):
        assert torch.equal(u, v)


@pytest.mark.parametrize("shape", [(1, 16), (5, 3, 528), (33, 28672)], ids=str)
def test_swiglu(shape):
    x = draw(*shape, seed=1, scale=2.0)
    g = draw(*shape[:-1], shape[-1] // 2, seed=2)

    def exact(t):
        a, b = t.chunk(2, -1)
        return torch.nn.functional.silu(a) * b

    check(grads(training.swiglu, [x], [g]), grads(training._swiglu, [x], [g]),
          grads(exact, [x], [g], torch.float64))


def steps():
    """Every fused step as a function of one bf16 tensor."""
    w = draw(768, seed=9, scale=0.2) + 1
    fused, plain, _ = attention(4, 1, 128, 9, 0)
    x = draw(2, 9, 768, seed=3)
    m = draw(1024, 768, seed=10, scale=768 ** -0.5)
    p = draw(4, 768, seed=11)
    return {"attention": (fused, plain, x),
            "norm": (lambda t: sum(training.norm(t, w, 1e-5)),
                     lambda t: t + training._rms(t, w, 1e-5), x),
            "swiglu": (training.swiglu, training._swiglu, x),
            "linear": (lambda t: training.linear(t, m),
                       lambda t: torch.nn.functional.linear(t, m), x),
            "prompts": (lambda t: training.add_prompts(t, p),
                        lambda t: training._add_prompts(t, p), x)}


@pytest.mark.parametrize("M,N,K", [(1, 32, 256), (33, 1056, 256), (127, 4096, 512),
                                   (128, 256, 256), (129, 2080, 512), (300, 3104, 768)])
@pytest.mark.parametrize("splits", [0, 1, 2, 7])
def test_gradient_of_a_projection(M, N, K, splits):
    """Rows that end within a tile, steps that do not share out evenly."""
    g, w = draw(M, N, seed=1), draw(N, K, seed=2, scale=N ** -0.5)
    got = training._ext().linear_grad(g, w, splits)
    want = g.double() @ w.double()
    # one rounding to bf16, eight significant bits: half a unit of the last one is
    # 2^-9 of the next power of two, up to 2^-8 of the value; products are exact in 32
    # bits, whose sums round N times
    tol = 2.0 ** -8 * want.abs() + N * 2.0 ** -24 * (g.double().abs()
                                                     @ w.double().abs())
    assert bool(((got.double() - want).abs() <= tol).all())


def test_projections_at_the_rule():
    """Sizes that a kernel takes forward, backward or both ways, and sizes left to torch."""
    for M, N, K, forward, backward in (
            (128, 256, 256, True, True), (129, 256, 256, True, True),
            (64, 264, 256, True, False), (64, 256, 320, True, False),
            (130, 1056, 256, True, True), (129, 288, 256, True, False),
            (32, 256, 256, False, True), (8, 264, 256, False, False),
            (64, 256, 264, False, False), (1, 2080, 512, False, True),
            (1025, 1024, 256, True, True)):
        assert ops.hip_ops.rows_wins(M, N, K) == forward
        assert training._split_gradient(M, N, K) == backward
        x, w = draw(M, K, seed=1), draw(N, K, seed=2, scale=K ** -0.5)
        g = draw(M, N, seed=3)
        taken = "_Linear" in type(training.linear(x.requires_grad_(True), w).grad_fn
                                  ).__name__
        assert taken == (forward or backward)
        f, p, e = (grads(fn, [x], [g], dt) for fn, dt in (
            (lambda t: training.linear(t, w), None),
            (lambda t: torch.nn.functional.linear(t, w), None),
            (lambda t: torch.nn.functional.linear(t, w.double()), torch.float64)))
        check(f, p, e)
    # gradients whose rows are not aligned, trained weights
    x, w = draw(4, 256).requires_grad_(True), draw(256, 256, seed=1)
    y = training.linear(x, w)
    off = draw(4 * 256 + 1, seed=2)[1:].view(4, 256)
    assert torch.equal(torch.autograd.grad(y, x, off)[0], off @ w)
    w.requires_grad_(True)
    assert torch.autograd.grad(training.linear(x, w).sum(), w)[0].shape == w.shape


@pytest.mark.parametrize("name", ["attention", "norm", "swiglu", "linear",
                                  "prompts"])
def test_watched_operations_stay_plain(name):
    """What looks into the operations gets the plain form's answer."""
    fused, plain, x = steps()[name]
    t = draw(*x.shape, seed=4)

    def same(a, b):
        # both bf16, a value of another order of rounding apart
        assert a.shape == b.shape
        assert away(a.float(), b.double()) < 0.02

    # gradients of gradients
    def twice(f):
        y = x.clone().requires_grad_(True)
        g, = torch.autograd.grad(f(y).float().square().sum(), y, create_graph=True)
        return torch.autograd.grad((g.float() * t.float()).sum(), y)[0]
    same(twice(fused), twice(plain))
    # a batch of gradients at once
    def batch(f):
        y = x.clone().requires_grad_(True)
        out = f(y)
        gs = torch.stack([draw(*out.shape, seed=s) for s in (5, 6)])
        return torch.autograd.grad(out, y, gs, is_grads_batched=True)[0]
    same(batch(fused), batch(plain))
    # forward mode, function transforms
    with torch.autograd.forward_ad.dual_level():
        d = [torch.autograd.forward_ad.unpack_dual(
            f(torch.autograd.forward_ad.make_dual(x, t))).tangent
            for f in (fused, plain)]
    same(*d)
    same(torch.func.vmap(fused)(x[None])[0], plain(x))
    same(*[torch.func.grad(lambda y: f(y).float().sum())(x) for f in (fused, plain)])
    # tracing
    same(torch.jit.trace(fused, x, check_trace=False)(x), plain(x))
    # saved tensors can be moved and come back
    y = x.clone().requires_grad_(True)
    with torch.autograd.graph.saved_tensors_hooks(lambda v: v.cpu(),
                                                  lambda v: v.to(DEV)):
        out = fused(y)
    z = x.clone().requires_grad_(True)
    ref = fused(z)
    g = draw(*out.shape, seed=7)
    assert torch.equal(torch.autograd.grad(out, y, g)[0],
                       torch.autograd.grad(ref, z, g)[0])
    # rows that do not lie one after the other
    wide = torch.cat([x, t], -1)[..., :x.shape[-1]]
    assert torch.equal(fused(wide), fused(x))


def test_trained_norm_weights_get_their_gradients():
    x, w = draw(3, 256), (draw(256, seed=1) + 1).requires_grad_(True)
    assert not training._fused(x, w)
    h, y = training.norm(x, w, 1e-5)
    assert torch.autograd.grad(y.sum(), w)[0].abs().sum() > 0


@pytest.mark.parametrize("B,T,n", [(1, 1, 1), (3, 7, 7), (2, 9, 4), (2, 5, 0)])
def test_prompts(B, T, n):
    x, p, g = draw(B, T, 264, seed=1), draw(n, 264, seed=2), draw(B, T, 264, seed=3)
    f, q, e = (grads(fn, [x, p], [g], dt) for fn, dt in (
        (training.add_prompts, None), (training._add_prompts, None),
        (training._add_prompts, torch.float64)))
    check(f, q, e)


@pytest.mark.parametrize("name", ["attention", "norm", "swiglu", "linear",
                                  "prompts"])
def test_rows_at_any_address(name):
    """Tensors that begin at two bytes into a line are read as they are elsewhere."""
    fused, _, x = steps()[name]

    def off(t):
        wide = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)
        wide[1:].copy_(t.reshape(-1))
        return wide[1:].view(t.shape)

    y = x.clone().requires_grad_(True)
    z = off(x).requires_grad_(True)
    assert z.data_ptr() % 16 == 2 and z.is_contiguous()
    a, b = fused(y), fused(z)
    g = draw(*a.shape, seed=7)
    assert torch.equal(a, b)
    want, = torch.autograd.grad(a, y, g)
    got, = torch.autograd.grad(b, z, off(g))
    # an unaligned gradient may take the library's product
    assert away(got, want.double()) < 2.0 ** -8


def test_bindings_refuse_unaligned_rows():
    ext = training._ext()
    _, _, x = steps()["attention"]
    wide = torch.empty(x.numel() + 1, dtype=x.dtype, device=DEV)
    odd = wide[1:].view(x.shape)
    cos, sin = (t.to(DEV) for t in ops.rope_cos_sin(128, 16))
    with pytest.raises(RuntimeError, match="aligned"):
        ext.rope_attention(odd, 4, 1, cos, sin, 0, 1.0, True)
    out, qk, o32, lse = ext.rope_attention(x, 4, 1, cos, sin, 0, 1.0, True)
    off = torch.empty(out.numel() + 1, dtype=x.dtype, device=DEV)[1:].view(out.shape)
    with pytest.raises(RuntimeError, match="aligned"):
        ext.rope_attention_grad(off, x, qk, o32, lse, 4, 1, cos, sin, 0, 1.0)


def test_another_device_than_the_current_one(monkeypatch):
    """The kernels go to the current device's stream: a tensor of another one takes
    the torch operations, which switch devices themselves."""
    forms = steps()
    assert all(f(x.clone().requires_grad_(True)).grad_fn is not None
               and training._fused(x) for f, _, x in forms.values())
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    for fused, plain, x in forms.values():
        assert not training._fused(x)
        y, z = (x.clone().requires_grad_(True) for _ in range(2))
        a, b = fused(y), plain(z)
        g = draw(*a.shape, seed=7)
        assert torch.equal(a, b)
        assert torch.equal(*(torch.autograd.grad(o, t, g)[0]
                             for o, t in ((a, y), (b, z))))


def test_function_modes_see_the_operations():
    class Watch(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    for name, (fused, plain, x) in steps().items():
        seen = []
        with Watch():
            fused(x)
        with Watch():
            mid, seen = seen, []
            plain(x)
        assert set(seen) <= set(mid), name
    # a default device replaces nothing
    with torch.device(DEV):
        assert training._fused(x)
