"""scatter_fused_runs_kernel (csrc/egs_scatter_fused.h) with the rows of a run of slices held in registers: from one unit of 32 picks
to as many as there are registers for and one more, few and many tokens, both weight layouts; against the oracle."""
import pytest
import torch

from oracle import egs_oracle as O
from tests._util import assert_close, make_case, np64
from tests.test_gpu_parity import dev

pytestmark = pytest.mark.gpu

from expertscattergather_amd import _abi
from expertscattergather_amd import hip_kernels as hk


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("shape", [
    (90, 5, 1, 3, 128, 32),         # one unit, fewer tokens than a wavefront sums at a time; in a run of two, not held
    (128, 5, 1, 3, 704, 32),        # in a run of eleven, held
    (33, 300, 16, 64, 288, 64),     # every register taken, three rounds of tokens, a short last run
    (33, 130, 33, 17, 288, 64),     # one unit more than there are registers for
    (40, 129, 31, 33, 256, 32),     # two units per expert, the second of one pick: too many
    (80, 128, 11, 90, 160, 64),     # three units per expert, wavefronts of four and five units
], ids=lambda s: "x".join(map(str, s)))
def test_held_rows_match_the_oracle(shape, dtype):
    B, T, E, K, I, J = shape
    case = make_case(sum(shape), *shape, dtype)
    Ind = torch.randint(0, T, (B, E, K), generator=torch.Generator().manual_seed(K))        # with repeats
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
