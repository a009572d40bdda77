"""A decode step of whole spans in one launch (ops/span.py): against 64 bits at the edges
of its slots, tiles and splits, with fewer workgroups than slots, beside another launch,
under capture, with what is not a number; and what is left to the blocks."""
import math

import pytest
import torch

from bloombee_amd.engine import BlockStack
from bloombee_amd.models.llama.config import LlamaConfig
from bloombee_amd.models.qwen3.config import Qwen3Config

DEV = "cuda:0"
gpu = pytest.mark.gpu


def stack(H, I, Hq, Hkv, layers, norms, device=DEV):
    cls = Qwen3Config if norms else LlamaConfig
    cfg = cls(hidden_size=H, intermediate_size=I, num_attention_heads=Hq,
              num_key_value_heads=Hkv, head_dim=128, num_hidden_layers=layers,
              vocab_size=64, max_position_embeddings=8192, rope_theta=10000.0)
    with torch.device(device):
        s = BlockStack(cfg, 0, layers, device=device)
    gen = torch.Generator(device).manual_seed(7)
    for blk in s.blocks:
        for name, w in blk.named_parameters():
            r = torch.randn(w.shape, generator=gen, device=device)
            w.data.copy_(1 + 0.1 * r if w.dim() == 1 else r / math.sqrt(w.shape[1]))
    return cfg, s


def session(s, lengths, page_size=16, room=None):
    """A filled session of sequences whose last token is the new one."""
    room = room or max(lengths)
    pool = s.make_kv(len(lengths) * (room + 32) + 64)
    kv = pool.allocate(len(lengths), room)
    kv.extend(room)
    gen = torch.Generator(DEV).manual_seed(3)
    for i in pool.own_layers:
        pool.k_pages(i).normal_(generator=gen)
        pool.v_pages(i).normal_(generator=gen)
    start = torch.tensor([n - 1 for n in lengths], dtype=torch.int32, device=DEV)
    return pool, kv, start


def rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def turn(x, pos, base):
    f = base ** (-torch.arange(64, device=DEV, dtype=torch.float64) / 64)
    a = pos.double()[:, None, None] * f
    u, v = x[..., :64], x[..., 64:]
    return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()], -1)


def exact(cfg, weights, x, pool, kv, start, pos):
    """The step in 64 bits: hidden states, new keys and values of each layer."""
    B, G = x.shape[0], cfg.num_key_value_heads
    Hq, P, eps = cfg.num_attention_heads, pool.page_size, cfg.rms_norm_eps
    table, x, new = kv.page_table().long(), x[:, 0].double(), []
    for i, w in enumerate(weights):
        qkv = rms(x, w["input_norm_w"], eps) @ w["qkv_w"].double().T
        q, k, v = qkv.view(B, -1, 128).split([Hq, G, G], 1)
        if "q_norm_w" in w:
            q, k = rms(q, w["q_norm_w"], eps), rms(k, w["k_norm_w"], eps)
        q, k = turn(q, pos, cfg.rope_theta), turn(k, pos, cfg.rope_theta)
        new.append((k, v))
        out = []
        for b in range(B):
            n = int(start[b])
            pages = table[b, :n // P + 1]
            kb = pool.k_pages(i)[pages].double().transpose(1, 2).flatten(0, 1)[:n]
            vb = pool.v_pages(i)[pages].double().permute(0, 3, 1, 2).flatten(0, 1)[:n]
            kb, vb = torch.cat([kb, k[b:b + 1]]), torch.cat([vb, v[b:b + 1]])
            for h in range(Hq):
                p = torch.softmax(kb[:, h * G // Hq] @ q[b, h] / math.sqrt(128), 0)
                out.append(p @ vb[:, h * G // Hq])
        x = x + torch.stack(out).view(B, -1) @ w["o_w"].double().T
        g, u = (rms(x, w["post_norm_w"], eps) @ w["gate_up_w"].double().T).chunk(2, -1)
        x = x + (torch.nn.functional.silu(g) * u) @ w["down_w"].double().T
    return x, new


def relative(a, b):
    return float((a.double() - b).norm() / b.norm())


def in_one_launch(s, monkeypatch):
    """Counts the steps that took one."""
    from bloombee_amd import engine
    taken, plain = [], engine.decode_span

    def spy(*args):
        out = plain(*args)
        taken.append(out is not None)
        return out
    monkeypatch.setattr(engine, "decode_span", spy)
    return taken


SMALL, QWEN, WIDE = (256, 512, 2, 1), (1024, 3072, 16, 8), (2048, 5632, 16, 4)


# sizes: fewer units than slots; pieces of K for some of the waves only; all registers of
# a small model, a unit more than they hold, groups of units; eight heads on a key head.
# lengths: ends of pages, tiles and splits, the first token, splits twice as long,
# splits that leave no slot for attention alone
@gpu
@pytest.mark.parametrize("sizes,norms", [
    (SMALL, False), ((768, 1280, 6, 2), True), (QWEN, True), ((1280, 3328, 10, 5), True),
    (WIDE, False), ((1536, 4352, 16, 2), False)])
@pytest.mark.parametrize("lengths", [
    [1], [32, 33], [256, 257, 17], [5, 300, 1, 700], [2100, 40, 3000, 700]])
def test_against_64_bits(sizes, norms, lengths, monkeypatch):
    layers = 2
    cfg, s = stack(*sizes, layers, norms)
    weights = [{n: w.detach().clone() for n, w in b.named_parameters()}
               for b in s.blocks]
    pool, kv, start = session(s, lengths)
    x = torch.randn(len(lengths), 1, sizes[0], device=DEV).bfloat16()
    before = [(pool.k_pages(i).clone(), pool.v_pages(i).clone()) for i in range(layers)]
    taken = in_one_launch(s, monkeypatch)
    want, new = exact(cfg, weights, x, pool, kv, start, start)
    got = s.forward_inference(x, kv, start)
    assert taken == [True]
    # eight roundings to bf16 a layer, of 2^-9 at most each, independent; norms folded
    # into weights round those once more
    bound = 2.0 ** -9 * math.sqrt(10 * layers)
    assert relative(got[:, 0], want) < bound
    P, table = pool.page_size, kv.page_table().long()
    for i, (k, v) in enumerate(before):
        at = start.long()
        page = table[torch.arange(len(lengths), device=DEV), at // P]
        assert relative(pool.k_pages(i)[page, :, at % P], new[i][0]) < bound
        assert relative(pool.v_pages(i)[page, :, :, at % P], new[i][1]) < bound
        # nothing else changes
        k[page, :, at % P] = pool.k_pages(i)[page, :, at % P]
        v[page, :, :, at % P] = pool.v_pages(i)[page, :, :, at % P]
        assert torch.equal(k, pool.k_pages(i)) and torch.equal(v, pool.v_pages(i))
    assert torch.equal(s.forward_inference(x, kv, start), got)


# more splits of a sequence than a wave has lanes, of a small model's slots for attention
# alone, of all slots, of a wide model; the values behind the 64th are unlike the others
@gpu
@pytest.mark.parametrize("sizes,lengths", [
    (SMALL, [16700]), (SMALL, [70001]), ((1536, 4352, 16, 2), [17001]),
    ((1024, 4096, 8, 1), [300, 20000])])
def test_many_splits(sizes, lengths, monkeypatch):
    cfg, s = stack(*sizes, 2, False)
    pool, kv, start = session(s, lengths)
    weights = [{n: w.detach().clone() for n, w in b.named_parameters()}
               for b in s.blocks]
    table = kv.page_table().long()
    for i in range(2):
        pool.v_pages(i)[table[len(lengths) - 1, 64 * 256 // 16:]] += 8
    x = torch.randn(len(lengths), 1, sizes[0], device=DEV).bfloat16()
    want, _ = exact(cfg, weights, x, pool, kv, start, start.clamp(max=8191))
    taken = in_one_launch(s, monkeypatch)
    got = s.forward_inference(x, kv, start)
    assert taken == [True]
    assert relative(got[:, 0], want) < 2.0 ** -9 * math.sqrt(10 * 2)


@gpu
@pytest.mark.parametrize("page", [8, 32])
def test_pages_and_positions(page, monkeypatch):
    """Other pages, positions that are not the places in the cache, more layers than
    a launch's arguments hold."""
    monkeypatch.setenv("BBAMD_KV_PAGE_SIZE", str(page))
    from bloombee_amd import config
    monkeypatch.setattr(config.get_config().kv, "page_size", page)
    cfg, s = stack(*SMALL, 50, True)
    pool, kv, start = session(s, [70, 9])
    assert pool.page_size == page
    weights = [{n: w.detach().clone() for n, w in b.named_parameters()}
               for b in s.blocks]
    x = torch.randn(2, 1, SMALL[0], device=DEV).bfloat16()
    pos = torch.tensor([[900], [9000]], dtype=torch.int64, device=DEV)
    want, _ = exact(cfg, weights, x, pool, kv, start, pos[:, 0].clamp(max=8191))
    taken = in_one_launch(s, monkeypatch)
    got = s.forward_inference(x, kv, start, pos)
    assert taken == [True]
    assert relative(got[:, 0], want) < 2.0 ** -9 * math.sqrt(10 * 50)


def arguments(s, x, kv, start):
    weights = []
    for i, b in enumerate(s.blocks):
        b.fold_norm_weights()
        weights += [b.qkv_w, b.o_w, b.gate_up_w, b.down_w, *b.span_norms(),
                    kv.k_pages(i), kv.v_pages(i)]
    cos, sin = s.blocks[0].rope.get(x.device)
    return (x, weights, s.blocks[0].Hq, cos, sin, None, start, kv.page_table(), 1e-5,
            0.09)


@gpu
@pytest.mark.parametrize("sizes,lengths", [(QWEN, [40, 300]), (WIDE, [500]),
                                           (SMALL, [1, 2, 3, 700])])
@pytest.mark.parametrize("groups", [1, 48, 255])
def test_fewer_workgroups_than_slots(sizes, lengths, groups):
    """Who waits takes up slots that nobody runs; the sums are the same."""
    from bloombee_amd.ops import span
    _, s = stack(*sizes, 2, True)
    _, kv, start = session(s, lengths)
    x = torch.randn(len(lengths), 1, sizes[0], device=DEV).bfloat16()
    args = arguments(s, x, kv, start)
    want = span._ext().decode_span(*args)
    assert torch.equal(span._ext().decode_span(*args, groups=groups), want)


@gpu
def test_beside_another_launch():
    """Two streams at once, on caches of their own."""
    from bloombee_amd.ops import span
    _, s = stack(*QWEN, 4, True)
    runs = []
    for n in (100, 900):
        _, kv, start = session(s, [n])
        x = torch.randn(1, 1, 1024, device=DEV).bfloat16()
        args = arguments(s, x, kv, start)
        runs.append((torch.cuda.Stream(), args, span._ext().decode_span(*args)))
    torch.cuda.synchronize()
    got = []
    for _ in range(10):
        for stream, args, want in runs:
            with torch.cuda.stream(stream):
                got.append((span._ext().decode_span(*args), want))
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in got)


@gpu
@pytest.mark.parametrize("sizes", [QWEN, WIDE], ids=["small", "wide"])
@pytest.mark.parametrize("cycles", [10 ** 5, 4 * 10 ** 5, 10 ** 6, 10 ** 7])
def test_beside_a_launch_that_stays(sizes, cycles):
    """A compute unit is held as long as a few layers, half of them, all: its slot's own
    workgroup comes to relieve who stands in, or too late."""
    from bloombee_amd.ops import span
    _, s = stack(*sizes, 12, True)
    _, kv, start = session(s, [40, 300])
    args = arguments(s, torch.randn(2, 1, sizes[0], device=DEV).bfloat16(), kv, start)
    want = span._ext().decode_span(*args)
    other = torch.cuda.Stream()
    torch.cuda.synchronize()
    got = []
    for _ in range(3):
        with torch.cuda.stream(other):
            torch.cuda._sleep(cycles)
        got.append(span._ext().decode_span(*args))
    torch.cuda.synchronize()
    assert all(torch.equal(g, want) for g in got)


@gpu
def test_replayed():
    """A captured step at other positions, eager steps in between."""
    _, s = stack(*QWEN, 3, True)
    _, kv, start = session(s, [600, 600], room=700)
    x = torch.randn(2, 1, 1024, device=DEV).bfloat16()
    s.forward_inference(x, kv, start)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = s.forward_inference(x, kv, start)
    for at in ([599, 599], [255, 256], [3, 640], [699, 31]):
        start.copy_(torch.tensor(at, dtype=torch.int32))
        x.normal_()
        want = s.forward_inference(x, kv, start).clone()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@gpu
def test_not_a_number():
    """A row of NaN with all bits set stays one, alone; infinities end as NaN."""
    _, s = stack(*QWEN, 2, True)
    _, kv, start = session(s, [30, 30, 30])
    x = torch.randn(3, 1, 1024, device=DEV).bfloat16()
    want = s.forward_inference(x, kv, start).clone()
    x[1] = torch.full((1, 1024), -1, dtype=torch.int16).view(torch.bfloat16).to(DEV)
    x[2, 0, 5] = math.inf
    got = s.forward_inference(x, kv, start)
    assert torch.equal(got[0], want[0])
    assert bool(got[1].isnan().all()) and bool(got[2].isnan().any())


@gpu
def test_left_to_the_blocks(monkeypatch):
    """Several tokens, five sequences, adapters, quantized weights, a step of one's own."""
    _, s = stack(*SMALL, 2, False)
    taken = in_one_launch(s, monkeypatch)

    def step(B=1, T=1):
        _, kv, start = session(s, [20 + T] * B)
        x = torch.randn(B, T, SMALL[0], device=DEV).bfloat16()
        s.forward_inference(x, kv, start - T + 1)
        n = taken.count(True)
        taken.clear()
        return n
    assert step() == 1 and step(4) == 1
    assert step(T=2) == 0 and step(5) == 0
    blk = s.blocks[1]
    blk.lora_delta = lambda name, x: None
    assert step() == 0
    del blk.lora_delta
    blk.forward_inference = type(blk).forward_inference.__get__(blk)
    assert step() == 0
    del blk.forward_inference
    blk.streamed, folded = True, blk._norm_folded
    blk._norm_folded = False
    assert step() == 0
    blk.streamed, blk._norm_folded = False, folded
    assert step() == 1
    blk.quantize_weights_q4(keep_full=True)
    assert step() == 0


@gpu
def test_sizes_are_asked_ahead_of_the_layers(monkeypatch):
    """Layers that no launch takes are not walked for it at each step."""
    cfg = LlamaConfig(hidden_size=512, intermediate_size=1024, num_attention_heads=8,
                      num_key_value_heads=2, head_dim=64, num_hidden_layers=6,
                      vocab_size=64, max_position_embeddings=64)
    s = BlockStack(cfg, 0, 6, device=DEV)
    taken = in_one_launch(s, monkeypatch)
    kv = s.make_kv(64).allocate(1, 32)
    kv.extend(9)
    asked = []
    pages = kv.k_pages
    monkeypatch.setattr(kv, "k_pages", lambda i: asked.append(i) or pages(i))
    s.forward_inference(torch.randn(1, 1, 512, device=DEV).bfloat16(), kv,
                        torch.tensor([8], dtype=torch.int32, device=DEV))
    assert not taken and asked == [0, 0, 1, 2, 3, 4, 5]


@pytest.mark.parametrize("change,fits", [
    ({}, True), (dict(M=4), True), (dict(M=5), False), (dict(M=0), False),
    (dict(D=64), False), (dict(P=16), True), (dict(P=4), False), (dict(P=12), False),
    (dict(Hq=24), True), (dict(Hq=20), False), (dict(Hq=72), False), (dict(H=1152), False),
    (dict(I=3200), False), (dict(H=4096, I=14336, Hq=32, M=2), True),
    (dict(H=4096, I=14336, Hq=32, M=3), False), (dict(Hkv=32, Hq=64, M=4), True),
    (dict(Hkv=128, Hq=128, M=4), False), (dict(H=16384, I=65536), False)])
def test_sizes(change, fits):
    from bloombee_amd.ops import interface, span
    if not interface.HAVE_HIP_OPS:
        pytest.skip("the extension is not built")
    sizes = dict(M=1, H=1024, I=3072, Hq=16, Hkv=8, D=128, P=8) | change
    assert span._ext().span_fits(*(sizes[n] for n in
                                   ("M", "H", "I", "Hq", "Hkv", "D", "P"))) == fits
