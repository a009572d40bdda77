"""How prompt attention shares out its keys: by those that there are, not by those that
the page table has room for (no device)."""
import pytest
import torch

from bloombee_amd import ops
from bloombee_amd.engine import BlockStack
from bloombee_amd.kv.paged import context_bound
from bloombee_amd.kv.views import SessionView
from bloombee_amd.models.base import resolve_config

from tests.test_prefill_attention import TWO_GROUPS


@pytest.mark.skipif(not ops.HAVE_HIP_OPS, reason="extension not built")
@pytest.mark.parametrize("tokens,keys,window,plan", [
    # no splits of one tile of keys; two groups of waves; splits as well; many splits; a
    # window's keys and no others
    (64, 64, 0, (1, 1)), (333, 333, 0, (1, 2)), (333, 1534, 0, (2, 2)),
    (64, 8192, 0, (16, 2)), (64, 8192, 64, (1, 1)), (64, 8192, 256, (1, 2)),
    (4096, 8192, 64, (1, 1))])
def test_plan(tokens, keys, window, plan):
    assert ops.hip_ops.prefill_plan(1, 32, 8, tokens, 128, 16, keys, False, window) == plan


@pytest.mark.skipif(not ops.HAVE_HIP_OPS, reason="extension not built")
@pytest.mark.parametrize("case", TWO_GROUPS, ids=str)
def test_sizes_of_two_groups(case):
    """What the device tests hold for two groups of waves has two."""
    B, Hq, Hkv, D, T, starts, room, window = case
    for tree in (False, True):
        if not (tree and (window or T > 128)):
            plan = ops.hip_ops.prefill_plan(B, Hq, Hkv, T, D, 16, room, tree, window)
            assert plan[1] == 2


def spy(monkeypatch):
    """What the steps say of their longest context."""
    said = []
    for name in ("attn_paged", "attn_paged_qkv"):
        def wrapped(*a, f=getattr(ops, name), **k):
            said.append(k.get("longest"))
            return f(*a, **k)
        monkeypatch.setattr(ops, name, wrapped)
    return said


@pytest.mark.parametrize("model", ["llama-tiny", "bloom-tiny", "falcon-tiny", "qwen3-tiny",
                                   "mixtral-tiny", "gemma4-tiny"])
def test_steps_know_their_context(model, monkeypatch):
    """Of a session's room of 64, a first prompt of 9, a turn of 5, a token."""
    cfg = resolve_config(model)
    stack = BlockStack(cfg, 0, 2, device="cpu")
    kv = stack.make_kv(256).allocate(2, 64)
    said = spy(monkeypatch)
    for n, longest in ((9, 9), (5, 14), (1, 0)):
        start = torch.full((2,), kv.lengths[0], dtype=torch.int32)
        kv.extend(n)
        stack.forward_inference(torch.zeros(2, n, cfg.hidden_size, dtype=cfg.dtype), kv,
                                start)
        assert said and set(said) == {longest}
        said.clear()


def test_bound_of_a_session_and_its_rows():
    kv = BlockStack(resolve_config("llama-tiny"), 0, 1, device="cpu").make_kv(256)
    kv = kv.allocate(3, 64)
    kv.extend_rows(0, 1, 7)
    kv.extend_rows(1, 3, 4, speculative=True)
    assert context_bound(kv, 4) == 7
    assert context_bound(SessionView(kv, 1, 3), 4) == 4
    assert context_bound(kv, 1) == 0 and context_bound(object(), 4) == 0
