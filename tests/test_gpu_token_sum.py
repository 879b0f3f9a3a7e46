"""token_sum_kernel (csrc/egs_token_sum.h) with a wavefront per token: tokens nobody picked first, last and in a row, tokens of one to
thirty-two picks (nine: one more than are on their way at a time), of more, and of more than sixty-four, fewer tokens than wavefronts,
one token to a wavefront and several; against the oracle."""
import pytest
import torch

from oracle import egs_oracle as O
from tests._util import assert_close, make_case, np64
from tests.test_gpu_parity import dev

pytestmark = pytest.mark.gpu

from expertscattergather_amd import _abi
from expertscattergather_amd import hip_kernels as hk


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("mode", ["deterministic", "atomic"])
@pytest.mark.parametrize("T, counts", [(60, [0, 0, 9, 1, 8, 0, 0, 0, 0, 17, 16, 32, 0, 3]), (60, [0, 33, 5, 64, 1]), (60, [0, 65, 0, 7, 130]), (3, [0, 2, 0]), (2, [40, 0])],
                         ids=["few", "some", "hot", "three", "two"])
def test_sums_of_neighbouring_tokens(T, counts, mode, dtype):
    E, I, J = 5, 261, 24
    picks = [t for t, n in enumerate(counts) for _ in range(n)]
    picks += [T] * (-len(picks) % E)                    # a token that does not exist
    order = torch.randperm(len(picks), generator=torch.Generator().manual_seed(len(picks)))
    Ind = torch.stack([torch.tensor(picks)[order], torch.tensor(picks)]).reshape(2, E, -1).contiguous()
    B, K = 2, Ind.shape[2]
    case = make_case(T + K, B, T, E, K, I, J, dtype)
    hk.set_scatter_mode(mode)
    try:
        with _abi.launch_log() as log:
            out = hk.expert_scatter_forward_call(dev(case["Y"]), dev(case["Ws"]), dev(Ind), T, torch.float32)
    finally:
        hk.set_scatter_mode("deterministic")
    if mode == "deterministic" or dtype != torch.float32:
        assert log.kernels[-1] == "token_sum_kernel", log.kernels
    Y = np64(case["Y"]) * (Ind < T).numpy()[..., None]
    if mode == "atomic" and dtype != torch.float32:     # product rows in the element type
        return assert_close(out.float(), O.scatter_forward(Y, np64(case["Ws"]), Ind.clamp(max=T - 1).numpy(), T), torch.bfloat16, "out")
    assert_close(out, O.scatter_forward(Y, np64(case["Ws"]), Ind.clamp(max=T - 1).numpy(), T), dtype, "out")


def test_several_tokens_to_a_wavefront():
    """1536 workgroups of four tokens would be more than a thousand: eight to a workgroup, two to a wavefront, of up to 64 picks."""
    B, T, E, K, I, J = 64, 96, 5, 40, 261, 24
    case = make_case(4, B, T, E, K, I, J, torch.float32)
    Ind = case["Ind"].clone()
    Ind[:, 0, :], Ind[:, 1, :20], Ind[1::2, 2, :] = 7, 7, 7              # 60 picks of a token, or a hundred
    with _abi.launch_log() as log:
        out = hk.expert_scatter_forward_call(dev(case["Y"]), dev(case["Ws"]), dev(Ind), T, torch.float32)
    assert log.kernels[-1] == "token_sum_kernel", log.kernels
    assert_close(out, O.scatter_forward(np64(case["Y"]), np64(case["Ws"]), Ind.numpy(), T), torch.float32, "out")
