"""segment_sum_kernel (csrc/egs_scatter_aux.h) at row lengths around its pieces of four columns and its groups of threads, tokens with no pick, with
fewer than a long segment's 64 and with several chunks of it; against the oracle, the same bits again."""
import pytest
import torch

from oracle import egs_oracle as O
from tests._util import assert_close, make_case, np64
from tests.test_gpu_parity import dev

pytestmark = pytest.mark.gpu

from expertscattergather_amd import _abi
from expertscattergather_amd import hip_kernels as hk


@pytest.mark.parametrize("mode", ["deterministic", "atomic"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("I", [1, 2, 3, 5, 26, 31, 33, 66, 129, 258, 510, 513, 1026])
def test_rows_of_any_length(I, dtype, mode):
    B, T, E, K, J = 2, 180, 69, 120, 19                 # 8280 picks: a routing table
    case = make_case(I, B, T, E, K, I, J, dtype)
    gen = torch.Generator().manual_seed(I)
    Ind = torch.randint(0, T - 1, (B, E, K), generator=gen)             # about 46 picks a token, the last token none
    Ind[0, :, :7] = 5                                   # 480 more: nine chunks
    Ind[1, 0, 0], Ind[1, 1, 1] = T, -1                  # picks that do not exist
    Ys = np64(case["Y"]) * ((Ind >= 0) & (Ind < T)).numpy()[..., None]
    want = O.scatter_forward(Ys, np64(case["Ws"]), Ind.clamp(0, T - 1).numpy(), T)
    with hk.scatter_mode_scope(mode):
        with _abi.launch_log() as log:
            out = hk.expert_scatter_forward_call(dev(case["Y"]), dev(case["Ws"]), dev(Ind), T, torch.float32)
        again = hk.expert_scatter_forward_call(dev(case["Y"]), dev(case["Ws"]), dev(Ind), T, torch.float32)
    if mode == "atomic" and dtype is torch.float32:     # fp32 atomics on the output: no table, no sums
        assert "segment_sum_kernel" not in log.kernels, log.kernels
        return assert_close(out, want, dtype, "out")
    assert "segment_sum_kernel" in log.kernels, log.kernels
    assert torch.equal(out, again) and (out[:, T - 1] == 0).all()
    if mode == "deterministic":
        return assert_close(out, want, dtype, "out")
    # 16-bit rows: each pick's row is rounded to the element type (relative 2^-8, 2^-11) before the fp32 sum, which is rounded once more; the sum of the
    # magnitudes bounds both.  (1e-6: values below the normal ones of f16.)
    most = O.scatter_forward(abs(Ys), abs(np64(case["Ws"])), Ind.clamp(0, T - 1).numpy(), T)
    assert (abs(np64(out) - want) <= 2.02 * 2.0 ** (-8 if dtype is torch.bfloat16 else -11) * most + 1e-6).all()
