"""Prompt attention over paged caches at the edges of its tiles: rows are (token,
head of the group) pairs, 128 a workgroup, keys come in tiles of 64 and are split
over workgroups where the rows leave the device idle."""
import pytest
import torch

from bloombee_amd import ops
from bloombee_amd.ops import reference as ref

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def paged(B, Hkv, D, P, lengths, room, seed):
    """Pages in random order, with large values beyond each sequence's end."""
    gen = torch.Generator().manual_seed(seed)
    maxp = -(-room // P)
    n = B * maxp + 3
    kp = torch.randn(n, Hkv, P, D, generator=gen).bfloat16()
    vp = torch.randn(n, Hkv, D, P, generator=gen).bfloat16()
    table = torch.randperm(n, generator=gen)[:B * maxp].view(B, maxp).int()
    for b, length in enumerate(lengths):
        for pos in range(length, maxp * P):
            page = int(table[b, pos // P])
            kp[page, :, pos % P] = 50.0
            vp[page, :, :, pos % P] = 50.0
    return kp, vp, table


CASES = [
    # B, Hq, Hkv, D, P, tokens, starts, room, window
    (1, 4, 2, 128, 16, 2, (0,), 16, 0),            # the smallest prompt
    (2, 8, 2, 128, 16, 25, (1500, 3), 1600, 0),    # split keys, one side short
    (1, 8, 8, 64, 16, 65, (63,), 128, 0),          # one row over a tile
    (1, 4, 1, 128, 16, 33, (95,), 128, 0),         # rows of 33 tokens, 132
    (1, 6, 2, 128, 8, 43, (21,), 64, 0),           # a group of three, small pages
    (2, 4, 4, 32, 32, 129, (0, 31), 160, 0),
    (1, 2, 1, 256, 16, 70, (130,), 256, 0),
    (8, 32, 8, 128, 16, 127, (0, 1, 2, 63, 64, 65, 7, 0), 192, 0),  # no splits
    (2, 8, 2, 128, 16, 100, (300, 0), 512, 64),    # a window of one tile
    (1, 4, 2, 64, 16, 90, (200,), 400, 33),
    (1, 71, 1, 64, 16, 5, (40,), 64, 0),           # a wide group
]


def close(got, want):
    # weights enter the value product in bf16 and the result is bf16: 2^-9 of the
    # largest value (4.5 standard deviations) each
    err = (got.cpu().float() - want.float()).abs().max()
    assert err <= 2 * 4.5 * 2.0 ** -9, err


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c[:6])))
@pytest.mark.parametrize("form", ["plain", "alibi", "tree"])
def test_prompt_attention(case, form):
    B, Hq, Hkv, D, P, T, starts, room, window = case
    if form == "tree" and window:
        pytest.skip("tree steps have no window")
    kp, vp, table = paged(B, Hkv, D, P, [s + T for s in starts], room, seed=T)
    gen = torch.Generator().manual_seed(3)
    q = torch.randn(B, Hq, T, D, generator=gen).bfloat16()
    qs = torch.tensor(starts, dtype=torch.int32)
    slopes = ops.alibi_slopes_for(Hq) if form == "alibi" else None
    tree = None
    if form == "tree":
        tree = torch.rand(B, T, T, generator=gen) < 0.3
        tree |= torch.eye(T, dtype=torch.bool)
    want = ref.attn_paged(q.float(), kp.float(), vp.float(), table, qs.long(),
                          sliding_window=window or None, alibi_slopes=slopes,
                          tree_mask=tree)
    dev = [t.to(DEV) for t in (q, kp, vp, table, qs)]
    got = ops.attn_paged(*dev, window=window, alibi_slopes=slopes,
                         tree_mask=None if tree is None else tree.to(DEV))
    close(got, want)


@pytest.mark.parametrize("case", CASES[1:5], ids=lambda c: "-".join(map(str, c[:6])))
def test_queries_of_a_fused_projection(case):
    """Queries read from [q | k | v] rows, results in rows of heads; infinite keys
    beyond the context do no harm."""
    B, Hq, Hkv, D, P, T, starts, room, window = case
    kp, vp, table = paged(B, Hkv, D, P, [s + T for s in starts], room, seed=T)
    kp[kp == 50.0] = float("inf")
    gen = torch.Generator().manual_seed(3)
    qkv = torch.randn(B, T, (Hq + 2 * Hkv) * D, generator=gen).bfloat16()
    qs = torch.tensor(starts, dtype=torch.int32)
    want = ops.attn_paged_qkv(qkv.float(), Hq, Hkv, kp.float(), vp.float(), table,
                              qs)
    got = ops.attn_paged_qkv(qkv.to(DEV), Hq, Hkv, kp.to(DEV), vp.to(DEV),
                             table.to(DEV), qs.to(DEV))
    close(got, want)


@pytest.mark.parametrize("case", [CASES[1], CASES[7]], ids=["split", "unsplit"])
@pytest.mark.parametrize("form", ["plain", "alibi"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")], ids=str)
@pytest.mark.parametrize("where", ["key", "query"])
def test_rows_without_a_finite_result_say_so(case, form, bad, where):
    """A row that meets a NaN or an infinite score is NaN whether its keys are split
    or not; rows that do not are as they were."""
    B, Hq, Hkv, D, P, T, starts, room, _ = case
    kp, vp, table = paged(B, Hkv, D, P, [s + T for s in starts], room, seed=T)
    gen = torch.Generator().manual_seed(3)
    q = torch.randn(B, Hq, T, D, generator=gen).bfloat16()
    if where == "key":                       # of one head, seen from the tenth token on
        pos = starts[0] + 9
        kp[int(table[0, pos // P]), 0, pos % P, 5] = bad
    else:
        q[0, 1, 7, 3] = bad
    qs = torch.tensor(starts, dtype=torch.int32)
    slopes = ops.alibi_slopes_for(Hq) if form == "alibi" else None
    want = ref.attn_paged(q.float(), kp.float(), vp.float(), table, qs.long(),
                          alibi_slopes=slopes)
    assert bool(want.isnan().any()) and bool(want.isfinite().any())
    got = ops.attn_paged(*[t.to(DEV) for t in (q, kp, vp, table, qs)],
                         alibi_slopes=slopes).cpu()
    assert torch.equal(got.isnan(), want.isnan())
    close(got.nan_to_num(0), want.nan_to_num(0))


@pytest.mark.parametrize("P", [24, 40, 4, 12])
@pytest.mark.parametrize("form", ["plain", "window", "alibi", "tree"])
@pytest.mark.parametrize("start", [3, 1500])
def test_pages_of_other_sizes(P, form, start):
    """Pages of eight times any number of keys, and others, for prompts and for one
    token."""
    B, Hq, Hkv, D, T = 2, 4, 2, 64, 37
    starts = (start, 17)
    kp, vp, table = paged(B, Hkv, D, P, [s + T for s in starts], 1600, seed=P)
    gen = torch.Generator().manual_seed(3)
    q = torch.randn(B, Hq, T, D, generator=gen).bfloat16()
    qs = torch.tensor(starts, dtype=torch.int32)
    slopes = ops.alibi_slopes_for(Hq) if form == "alibi" else None
    tree = None
    if form == "tree":
        tree = torch.rand(B, T, T, generator=gen) < 0.3
        tree |= torch.eye(T, dtype=torch.bool)
    window = 50 if form == "window" else 0
    want = ref.attn_paged(q.float(), kp.float(), vp.float(), table, qs.long(),
                          sliding_window=window or None, alibi_slopes=slopes,
                          tree_mask=tree)
    got = ops.attn_paged(*[t.to(DEV) for t in (q, kp, vp, table, qs)], window=window,
                         alibi_slopes=slopes,
                         tree_mask=None if tree is None else tree.to(DEV))
    close(got, want)
    if tree is None:
        last = [t.to(DEV) for t in (q[:, :, -1:], kp, vp, table, qs + T - 1)]
        close(ops.attn_paged(*last, window=window, alibi_slopes=slopes),
              want[:, :, -1:])
    # and with queries of a fused projection
    if form != "alibi":
        qkv = torch.zeros(B, T, (Hq + 2 * Hkv) * D, dtype=torch.bfloat16)
        qkv[..., :Hq * D] = q.transpose(1, 2).reshape(B, T, -1)
        got = ops.attn_paged_qkv(qkv.to(DEV), Hq, Hkv, kp.to(DEV), vp.to(DEV),
                                 table.to(DEV), qs.to(DEV), window=window,
                                 tree_mask=None if tree is None else tree.to(DEV))
        close(got.view(B, T, Hq, D).transpose(1, 2), want)


def test_pages_at_any_address():
    """Pages that begin at two bytes into a line are read as they are elsewhere."""
    B, Hq, Hkv, D, P, T, starts, room, _ = CASES[1]
    kp, vp, table = paged(B, Hkv, D, P, [s + T for s in starts], room, seed=T)
    q = torch.randn(B, Hq, T, D, generator=torch.Generator().manual_seed(3)).bfloat16()
    qs = torch.tensor(starts, dtype=torch.int32)

    def off(t):
        wide = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)
        wide[1:].copy_(t.reshape(-1))
        assert wide[1:].data_ptr() % 16 == 2
        return wide[1:].view(t.shape)

    q, kp, vp, table, qs = (t.to(DEV) for t in (q, kp, vp, table, qs))
    want = ops.attn_paged(q, kp, vp, table, qs)
    assert torch.equal(ops.attn_paged(q, off(kp), off(vp), table, qs), want)
    assert torch.equal(ops.attn_paged(off(q), kp, vp, table, qs), want)


@pytest.mark.parametrize("Hkv,D,room,tokens,start", [
    (2, 128, 64, 1, 36), (2, 128, 2000, 1, 1500),      # one token: one split, several
    (2, 64, 64, 25, 12), (2, 128, 2000, 25, 1476),     # a prompt: the same
    (8, 128, 64, 600, 5), (1, 256, 64, 3, 40),
])
def test_infinite_values_of_the_last_key(Hkv, D, room, tokens, start):
    """Places beyond the context take no part, also where an infinite value is near:
    whoever sees it has an infinite result."""
    room = max(room, start + tokens + 3)
    kp, vp, table = paged(1, Hkv, D, 16, [start + tokens], room, seed=5)
    last = start + tokens - 1
    vp[int(table[0, last // 16]), 0, 7, last % 16] = float("inf")
    q = torch.randn(1, 2 * Hkv, tokens, D,
                    generator=torch.Generator().manual_seed(3)).bfloat16()
    qs = torch.tensor([start], dtype=torch.int32)
    want = ref.attn_paged(q.float(), kp.float(), vp.float(), table, qs.long())[:, :, -1]
    assert int(want.isinf().sum()) == 2 and not bool(want.isnan().any())
    got = ops.attn_paged(*[t.to(DEV) for t in (q, kp, vp, table, qs)]).cpu()[:, :, -1]
    assert torch.equal(got.float().isinf(), want.isinf())
    seen = want.isfinite()
    close(got[seen], want[seen])


@pytest.mark.parametrize("D", [32, 64, 128, 256])
@pytest.mark.parametrize("P", [8, 16, 32, 128, 48])
@pytest.mark.parametrize("length", [63, 65, 200])
def test_pages_behind_the_last_key(D, P, length):
    """Every head size with pages that a wave or a lane looks up, tiles that end within a
    page and before it; keys that are not numbers behind the last one do no harm."""
    B, Hq, Hkv, T = 2, 4, 2, 37
    starts = (length - T, 1)
    kp, vp, table = paged(B, Hkv, D, P, [s + T for s in starts], 256, seed=P)
    kp[kp == 50.0] = float("nan")
    gen = torch.Generator().manual_seed(3)
    q = torch.randn(B, Hq, T, D, generator=gen).bfloat16()
    qs = torch.tensor(starts, dtype=torch.int32)
    want = ref.attn_paged(q.float(), kp.float().nan_to_num(0), vp.float(), table,
                          qs.long())
    close(ops.attn_paged(*[t.to(DEV) for t in (q, kp, vp, table, qs)]), want)


GROUPED = [
    # sizes at which two groups of waves share out a workgroup's keys: unsplit and split,
    # an odd number of tiles, nothing left for the second group, rows of both sides
    (1, 32, 8, 128, 300, (0,), 320, 0),
    (2, 32, 8, 128, 200, (500, 3), 704, 0),
    (1, 8, 2, 64, 128, (1000,), 4096, 0),
    (1, 8, 2, 128, 100, (0,), 2048, 0),
    (2, 32, 8, 32, 97, (411, 900), 1024, 0),
    (1, 32, 8, 128, 333, (400,), 752, 150),
]

# and those at which the rule takes two for certain, trees among them: every head size,
# unsplit and split, the second group with and without keys, a window
TWO_GROUPS = [
    (1, 16, 16, 128, 20, (300,), 320, 0),
    (1, 16, 16, 32, 33, (2001,), 2064, 0),
    (2, 16, 16, 64, 33, (1007, 3), 1040, 0),
    (2, 32, 8, 128, 60, (3, 980), 1040, 0),
    (1, 32, 8, 128, 333, (400,), 752, 400),
]


@pytest.mark.parametrize("case", GROUPED + TWO_GROUPS,
                         ids=lambda c: "-".join(map(str, c[:6])))
@pytest.mark.parametrize("form", ["plain", "alibi", "tree", "nan"])
def test_two_groups_of_waves(case, form):
    B, Hq, Hkv, D, T, starts, room, window = case
    if form == "tree" and (window or T > 128):
        pytest.skip("large trees have one group, and no window")
    P = 16
    kp, vp, table = paged(B, Hkv, D, P, [s + T for s in starts], room, seed=T)
    gen = torch.Generator().manual_seed(3)
    q = torch.randn(B, Hq, T, D, generator=gen).bfloat16()
    qs = torch.tensor(starts, dtype=torch.int32)
    slopes = ops.alibi_slopes_for(Hq) if form == "alibi" else None
    tree = None
    if form == "tree":
        tree = torch.rand(B, T, T, generator=gen) < 0.3
        tree |= torch.eye(T, dtype=torch.bool)
    if form == "nan":             # a key of each half, each of another head's
        for head, pos in ((0, starts[0] + 9), (1, starts[0] + T - 20)):
            kp[int(table[0, pos // P]), head, pos % P, 5] = float("nan")
    want = ref.attn_paged(q.float(), kp.float(), vp.float(), table, qs.long(),
                          sliding_window=window or None, alibi_slopes=slopes,
                          tree_mask=tree)
    got = ops.attn_paged(*[t.to(DEV) for t in (q, kp, vp, table, qs)], window=window,
                         alibi_slopes=slopes,
                         tree_mask=None if tree is None else tree.to(DEV)).cpu()
    assert torch.equal(got.isnan(), want.isnan())
    assert bool(want.isnan().any()) == (form == "nan")
    close(got.nan_to_num(0), want.nan_to_num(0))


@pytest.mark.parametrize("D", [32, 64, 128, 256])
@pytest.mark.parametrize("splits,starts", [(2, (254, 0)), (3, (382, 60)), (4, (510, 3)),
                                           (5, (638, 300)), (8, (1022, 100)),
                                           (9, (1150, 0)), (16, (2046, 700))])
def test_folds_of_any_number_of_splits(D, splits, starts):
    """One chunk of the fold, a chunk and a split, several; a context that leaves splits
    without keys."""
    B, Hq, Hkv, T, P, room = 2, 8, 2, 2, 16, starts[0] + 2
    assert ops.hip_ops.prefill_plan(B, Hq, Hkv, T, D, P, room, False, 0)[0] == splits
    kp, vp, table = paged(B, Hkv, D, P, [s + T for s in starts], room, seed=splits)
    gen = torch.Generator().manual_seed(3)
    q = torch.randn(B, Hq, T, D, generator=gen).bfloat16()
    qs = torch.tensor(starts, dtype=torch.int32)
    want = ref.attn_paged(q.float(), kp.float(), vp.float(), table, qs.long())
    got = ops.attn_paged(*[t.to(DEV) for t in (q, kp, vp, table, qs)])
    close(got, want)
