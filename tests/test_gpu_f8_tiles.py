"""rows_gemm_f8_kernel in 128 x 128 tiles (csrc/egs_rows_gemm_f8.h): the edges of rows, columns and slabs against the quantised oracle,
and the bits of the 256 x 256 tiles."""
import numpy as np
import pytest
import torch

from expertscattergather_amd import _abi
from expertscattergather_amd import hip_kernels as hk
from expertscattergather_amd import workloads as wl
from oracle import egs_oracle as O
from tests._util import assert_close, make_case
from tests.test_gpu_parity import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 5, 1, 1, 128, 16), (1, 300, 3, 127, 128, 112), (1, 300, 9, 128, 256, 128), (3, 90, 10, 43, 384, 144),
                                   (2, 200, 17, 129, 1280, 272)], ids=str)
def test_small_tiles_match_the_quantised_oracle(shape):
    B, T, E, K, I, J = shape
    case = make_case(47, B, T, E, K, I, J, torch.bfloat16)
    case["Ind"][0, 0, 0] = T                                 # contributes a zero row
    case["Ind"][-1, -1, -1] = -1
    Wq, scale = wl.quantize_fp8_weights(case["Wg"].float())
    with _abi.launch_log() as log:
        Y = hk.expert_gather_fp8_forward(dev(case["X"]), dev(Wq), dev(scale), dev(case["Ind"]))
    assert log.kernels[-1] == "rows_gemm_f8_kernel<128>", log.kernels
    ind = case["Ind"].numpy().astype(np.int64)
    live = (ind >= 0) & (ind < T)
    ref = O.gather_forward_fp8(case["X"].float().numpy(), Wq.view(torch.uint8).numpy(), scale.numpy(), np.where(live, ind, 0)) * live[..., None]
    assert_close(Y, ref, torch.bfloat16, "fp8 tiles")


def test_small_and_large_tiles_give_the_same_bits():
    """All 64 experts at once take the 256 x 256 tiles, eight of them at a time the small ones."""
    case = make_case(48, 20, 300, 64, 50, 1152, 496, torch.bfloat16)
    Wq, scale = wl.quantize_fp8_weights(case["Wg"].float())
    X, q, sc, ind = dev(case["X"]), dev(Wq), dev(scale), dev(case["Ind"])
    with _abi.launch_log() as log:
        Y = hk.expert_gather_fp8_forward(X, q, sc, ind)
    assert log.kernels[-1] == "rows_gemm_f8_kernel<256>", log.kernels
    for e in range(0, 64, 8):
        with _abi.launch_log() as log:
            part = hk.expert_gather_fp8_forward(X, q[e:e + 8].contiguous(), sc[e:e + 8].contiguous(), ind[:, e:e + 8].contiguous())
        assert log.kernels[-1] == "rows_gemm_f8_kernel<128>", log.kernels
        assert torch.equal(Y[:, e:e + 8], part)


@pytest.mark.parametrize("width", [128, 512, 640, 1024, 2176, 4096, 4224])
def test_row_quantiser_at_every_number_of_chunks_a_lane_holds(width):
    """quantize_rows_e4m3_kernel<1, 2, 4, 8, 0>: bit for bit the oracle's, also for zero rows and rows with a NaN or an infinity."""
    case = make_case(49, 2, 33, 2, 3, width, 16, torch.bfloat16)
    X = case["X"]
    X[0, 0] = 0
    X[1, 2, width - 1] = 1000                                # the largest value in the last lane's chunk
    Wq, scale = wl.quantize_fp8_weights(case["Wg"].float())
    run = lambda x: hk.expert_gather_fp8_forward(dev(x), dev(Wq), dev(scale), dev(case["Ind"]), return_quantised=True)[1:]
    Xq, xs = run(X)
    q_o, xs_o = O.quantize_rows_e4m3(X.float().numpy())
    assert np.array_equal(xs.cpu().numpy(), xs_o)
    assert np.array_equal(Xq.cpu().view(torch.uint8).numpy(), q_o)
    X[0, 1, width - 1], X[1, 3, 0] = float("nan"), float("-inf")
    xs = run(X)[1].cpu().reshape(2, 33)
    assert xs[0, 1].isnan() and xs[1, 3].isnan() and int(xs.isnan().sum()) == 2
