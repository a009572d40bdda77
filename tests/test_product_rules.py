"""Which products the kernels take, as the rules themselves say it (no device)."""
import pytest

from bloombee_amd import ops

pytestmark = pytest.mark.skipif(not ops.HAVE_HIP_OPS, reason="extension not built")


def grad_wins(M, N, K):
    from bloombee_amd.ops import training
    return training._ext().linear_grad_wins(M, N, K)


@pytest.mark.parametrize("K", [256, 1024, 4096])
@pytest.mark.parametrize("M", [1, 32, 33, 64, 3000])
def test_weights_without_rows_stay_torchs(M, K):
    h = ops.hip_ops
    assert not (h.rows_wins(M, 0, K) or h.rows_swiglu_wins(M, 0, K)
                or h.few_sums(M, 0, K) or grad_wins(M, 0, K))


@pytest.mark.parametrize("N,K,splits", [
    (8192, 28672, 4), (7168, 28672, 4), (8192, 16384, 3), (4096, 8192, 8),
    (4096, 14336, 4), (8192, 8192, 2), (5120, 13824, 3), (512, 14336, 16), (16384, 4096, 1)])
def test_splits_begin_in_channels_of_their_own(N, K, splits):
    """Up to 32 rows: splits fill the chip, but do not begin a multiple of 4 KiB apart
    where rows of W do (two of up to 8192 columns may)."""
    assert ops.hip_ops.few_splits(N, K) == splits


@pytest.mark.parametrize("M,N,K", [(33, 8192, 8192), (64, 8192, 8192), (80, 8192, 8192),
                                   (128, 8192, 8192), (33, 14336, 4096), (64, 16384, 4096),
                                   (48, 12288, 12288), (112, 8192, 4096)])
def test_tiles_begin_in_channels_of_their_own(M, N, K):
    tile, splits = ops.hip_ops.rows_plan(M, N, K, False)
    stages = K // (128 if tile == 9 else 64)     # the last tile takes twice the columns
    columns = -(-stages // splits) * K // stages
    assert splits == 1 or columns % 2048


@pytest.mark.parametrize("M,N,K,tiles", [
    (9, 4096, 8192, False), (12, 4096, 14336, False), (13, 4096, 14336, True),
    (9, 12288, 16384, False), (12, 8192, 28672, False), (17, 8192, 28672, True),
    (9, 10240, 8192, True), (8, 10240, 8192, False), (1, 5120, 13824, True)])
def test_some_rows_with_long_sums(M, N, K, tiles):
    assert ops.hip_ops.few_sums(M, N, K) == tiles


@pytest.mark.parametrize("M,N,K,plan", [
    (193, 6144, 4096, (6, 2)), (300, 4672, 4544, (6, 2)), (288, 18176, 4544, (1, 1)),
    (617, 1024, 2048, (9, 1))])
def test_low_tiles_cost_what_they_take_from_memory(M, N, K, plan):
    """Where the two lowest tiles looked the cheapest and were not."""
    assert ops.hip_ops.rows_plan(M, N, K, False) == plan


@pytest.mark.parametrize("M,N,K,wins", [
    (1, 64, 256, True), (1, 96, 256, False), (1, 64, 320, False),       # N % 64, K % 256
    (512, 4096, 16384, True), (513, 4096, 16384, True), (519, 4096, 16384, False),
    (512, 28672, 8192, True), (513, 57344, 8192, False), (638, 28672, 8192, True),
    (639, 28672, 8192, False),                                          # M * K * N
    (1024, 57344, 4096, True), (1025, 57344, 4096, False), (1024, 16384, 4096, True),
    (2999, 4096, 4096, False), (3000, 4096, 4096, True),
    (3599, 12288, 4096, False), (3600, 12288, 4096, True)])
def test_gradients_at_the_rule(M, N, K, wins):
    assert grad_wins(M, N, K) == wins


@pytest.mark.parametrize("M,N,K,wins", [
    (128, 288, 256, True), (129, 288, 256, False), (128, 256, 256, False),
    (1024, 28704, 4096, True), (1025, 28704, 4096, False), (1024, 28704, 5120, False),
    (128, 224, 256, False), (129, 1056, 256, True), (64, 96, 320, False)])
def test_gradients_of_32_rows_at_the_rule(M, N, K, wins):
    from bloombee_amd.ops import training
    assert training._half_steps(M, N, K) == wins


@pytest.mark.parametrize("M,N,K,wins", [
    (32, 256, 256, False), (33, 256, 256, True), (64, 252, 256, False),
    (64, 256, 192, False), (64, 256, 288, False), (384, 29160, 4096, True),
    (384, 29168, 4096, False), (385, 15576, 4096, True), (385, 15592, 4096, False),
    (512, 64, 16448, True), (513, 64, 16448, False), (513, 64, 16384, True)])
def test_products_at_the_rule(M, N, K, wins):
    assert ops.hip_ops.rows_wins(M, N, K) == wins
