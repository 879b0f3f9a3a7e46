"""dw_reduce4_kernel (csrc/egs_small.h): every number of partial sums that its batches of eight, four, two and one make; against the oracle."""
import pytest
import torch

from expertscattergather_amd import _abi
from expertscattergather_amd import hip_kernels as hk
from oracle import egs_oracle as O
from tests._util import assert_close, make_case, np64
from tests.test_gpu_parity import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits", [2, 3, 4, 5, 8, 9, 10, 12, 16, 17, 24, 63])
def test_partial_sums_match_the_oracle(splits):
    """One expert of 16 x 8, 128 picks a split."""
    case = make_case(splits, splits, 1300, 1, 128, 16, 8, torch.bfloat16)
    with _abi.launch_log() as log:
        _, dW = hk.expert_gather_backward_call(dev(case["X"]), dev(case["Wg"]), dev(case["Ind"]), dev(case["Y"]), torch.float32)
    assert any("dw" in k and "reduce" in k for k in log.kernels), log.kernels
    ref = O.gather_backward(np64(case["X"]), np64(case["Wg"]), case["Ind"].numpy(), np64(case["Y"]))[1]
    assert_close(dW, ref, torch.bfloat16, "dW")
