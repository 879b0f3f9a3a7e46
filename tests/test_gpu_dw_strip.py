"""dw_strip_kernel (csrc/egs_dw_strip.h): each of its tile widths with ragged last tiles, one pick more and less than slabs and offset
tables hold, splits, both layouts, picks that do not exist, strided rows; against the oracle."""
import pytest
import torch

from oracle import egs_oracle as O
from tests._util import assert_close, make_case, np64
from tests.test_gpu_parity import dev

pytestmark = pytest.mark.gpu

from expertscattergather_amd import _abi
from expertscattergather_amd import hip_kernels as hk


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("shape", [
    (1, 150, 5, 129, 136, 8),       # two slabs, the second of one pick; eight columns
    (16, 40, 3, 8, 200, 56),        # one slab; fewer workgroups than XCDs
    (9, 300, 60, 57, 640, 48),      # 96 columns, seven tiles, the last of 64; four slabs and one pick
    (41, 64, 64, 50, 384, 64),      # 96 columns, a second table of offsets two picks long
    (17, 140, 64, 130, 488, 64),    # four tiles of 128 columns, the last of 104; three tables of offsets
    (40, 100, 2, 100, 264, 64),     # splits
    (6, 200, 20, 150, 328, 136),    # 96 columns by three column tiles, the last of eight
    (18, 80, 60, 115, 512, 120),    # 128 by 128, ragged; slabs of 64, a second table of offsets 22 picks long
    (5, 300, 3, 200, 120, 200),     # few rows; splits
], ids=lambda s: "x".join(map(str, s)))
def test_strips_match_the_oracle(shape, dtype):
    B, T, E, K, I, J = shape
    case = make_case(sum(shape), *shape, dtype)
    Ind = case["Ind"].clone()
    Ind[0, 0, 0], Ind[-1, -1, -1] = T, -1               # picks that do not exist
    keep = ((Ind >= 0) & (Ind < T)).numpy()[..., None]
    safe = Ind.clamp(0, T - 1).numpy()
    X = torch.full((B, T + 3, I + 8), float("nan"), dtype=dtype)       # rows apart, NaN between them
    X[:, :T, :I] = case["X"]
    X = dev(X)[:, :T, :I]
    with _abi.launch_log() as log:
        _, dWg = hk.expert_gather_backward_call(X, dev(case["Wg"]), dev(Ind), dev(case["Y"]), torch.float32)
        _, dWs = hk.expert_scatter_backward_call(dev(case["Y"]), dev(case["Ws"]), dev(Ind), dev(case["dOut"]), torch.float32)
    assert log.kernels.count("dw_strip_kernel") == 2, log.kernels
    Y = np64(case["Y"]) * keep
    assert_close(dWg, O.gather_backward(np64(case["X"]), np64(case["Wg"]), safe, Y)[1], dtype, "dW of the gather")
    assert_close(dWs, O.scatter_backward(Y, np64(case["Ws"]), safe, np64(case["dOut"]))[1], dtype, "dW of the scatter")


@pytest.mark.parametrize("shape, kernels", [((12, 300, 15, 21, 192, 64), ["scatter_fused_dwtile_kernel"]),                      # 180 tiles of 32 x 32 in the scatter's launch
                                            ((50, 45, 16, 45, 160, 64), ["scatter_fused_dwtile_kernel"]),
                                            ((64, 60, 30, 32, 768, 64), ["scatter_fused_runs_kernel", "dw_strip_kernel"]),      # a scatter in runs shares none
                                            ((44, 60, 46, 80, 32, 192), ["tiled_dw_kernel", "tiled_dw_sum_kernel"])], ids=lambda s: "x".join(map(str, s)) if isinstance(s, tuple) else None)
def test_where_strips_are_not_taken(shape, kernels):
    B, T, E, K, I, J = shape
    case = make_case(sum(shape), *shape, torch.bfloat16)
    with _abi.launch_log() as log:
        _, dW = hk.expert_gather_backward_call(dev(case["X"]), dev(case["Wg"]), dev(case["Ind"]), dev(case["Y"]), torch.float32)
    assert log.kernels[-len(kernels):] == kernels, log.kernels
    assert_close(dW, O.gather_backward(np64(case["X"]), np64(case["Wg"]), case["Ind"].numpy(), np64(case["Y"]))[1], torch.bfloat16, "dW")
