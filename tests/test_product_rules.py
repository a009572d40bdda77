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
