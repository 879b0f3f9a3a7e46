"""scatter_fused_runs_kernel (csrc/egs_scatter_fused.h): several column slices per workgroup, with a last run that is shorter;
against the oracle."""
import pytest
import torch

from oracle import egs_oracle as O
from tests._util import assert_close, make_case, np64
from tests.test_gpu_parity import dev

pytestmark = pytest.mark.gpu

from expertscattergather_amd import _abi
from expertscattergather_amd import hip_kernels as hk


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("shape", [(37, 40, 4, 9, 288, 32), (64, 33, 9, 40, 256, 64), (140, 20, 5, 33, 192, 32)], ids=lambda s: "x".join(map(str, s)))
def test_runs_of_slices_match_the_oracle(shape, dtype):
    B, T, E, K, I, J = shape
    case = make_case(sum(shape), *shape, dtype)
    Ind = case["Ind"].clone()
    Ind[0, 0, 0], Ind[-1, -1, -1] = T, -1               # picks that do not exist
    keep = ((Ind >= 0) & (Ind < T)).numpy()[..., None]
    safe = Ind.clamp(0, T - 1).numpy()
    with _abi.launch_log() as log:
        out = hk.expert_scatter_forward_call(dev(case["Y"]), dev(case["Ws"]), dev(Ind), T, torch.float32)
        dX, _ = hk.expert_gather_backward_call(dev(case["X"]), dev(case["Wg"]), dev(Ind), dev(case["Y"]), torch.float32)
    assert log.kernels.count("scatter_fused_runs_kernel") == 2, log.kernels
    Y = np64(case["Y"]) * keep
    assert_close(out, O.scatter_forward(Y, np64(case["Ws"]), safe, T), dtype, "out")
    assert_close(dX, O.gather_backward(np64(case["X"]), np64(case["Wg"]), safe, Y)[0], dtype, "dX")
