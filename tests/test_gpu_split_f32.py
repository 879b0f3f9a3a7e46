"""The fp32 weight gradient on the bf16 matrix instruction (csrc/egs_split_f32.h): edges of its tiles, slabs and splits, operands that end
in the middle of a chunk, values that three bf16 pieces cannot hold, and its error against the fp32 instruction's; against the oracle."""
import numpy as np
import pytest
import torch

from oracle import egs_oracle as O
from tests._util import assert_close, make_case, np64
from tests.test_gpu_parity import dev

pytestmark = pytest.mark.gpu

from expertscattergather_amd import _abi
from expertscattergather_amd import hip_kernels as hk


def gradients(case, Ind, X, Y):
    with _abi.launch_log() as log:
        _, dWg = hk.expert_gather_backward_call(X, dev(case["Wg"]), Ind, Y, torch.float32)
        _, dWs = hk.expert_scatter_backward_call(Y, dev(case["Ws"]), Ind, dev(case["dOut"]), torch.float32)
    return dWg, dWs, log.kernels


@pytest.mark.parametrize("shape, splits", [((8, 40, 4, 128, 64, 64), True),         # whole tiles and slabs; 1024 picks
                                           ((8, 40, 3, 65, 65, 63), True),          # one past a tile, one short of one; 520 picks
                                           ((5, 30, 2, 103, 129, 1), True),         # 515 picks, a column tile of one column
                                           ((3, 50, 150, 33, 70, 130), False),      # 99 picks: four slabs, the last of three; 900 tiles
                                           ((16, 9, 320, 4, 3, 5), False),          # 64 picks per expert; rows shorter than a chunk
                                           ((26, 33, 48, 20, 66, 64), True)], ids=lambda s: "x".join(map(str, s)) if isinstance(s, tuple) else None)
def test_weight_gradient_of_split_floats(shape, splits):
    B, T, E, K, I, J = shape
    case = make_case(sum(shape), *shape, torch.float32)
    Ind, Y = case["Ind"].clone(), case["Y"].clone()
    if B * K > 1:
        Ind[0, 0, 0], Ind[-1, -1, -1] = T, -1
        Y[0, 0, 0] = Y[-1, -1, -1] = float("nan")               # picks that do not exist do not count, whatever their rows hold
    dWg, dWs, kernels = gradients(case, dev(Ind), dev(case["X"]), dev(Y))
    assert kernels.count("tiled_dw_split_kernel") == 2 and ("tiled_dw_sum_kernel" in kernels) == splits, kernels
    safe, Yk = Ind.clamp(0, T - 1).numpy(), np64(Y)
    if B * K > 1:
        Yk[0, 0, 0] = Yk[-1, -1, -1] = 0
    for got, want, what in ((dWg, O.gather_backward(np64(case["X"]), np64(case["Wg"]), safe, Yk)[1], "dWg"),
                            (dWs, O.scatter_backward(Yk, np64(case["Ws"]), safe, np64(case["dOut"]))[1], "dWs")):
        assert_close(got, want, torch.float32, what)
        # no worse than one rounding of the sum per product of a pick: 2^-24 sqrt(picks) of the result, times four
        assert np.sqrt(((np64(got) - want) ** 2).mean()) <= 4 * 2.0 ** -24 * max(1, B * K) ** 0.5 * np.sqrt((want ** 2).mean()), what


def test_views_that_end_in_the_middle_of_a_chunk():
    B, T, E, K, I, J = 9, 21, 6, 60, 37, 29
    case = make_case(5, B, T, E, K, I, J, torch.float32)
    wide = torch.full((B * T * 41,), float("nan"), device="cuda")
    X = wide[wide.numel() - ((B - 1) * T * 41 + (T - 1) * 41 + I):].as_strided((B, T, I), (T * 41, 41, 1))
    X.copy_(case["X"])
    dWg, dWs, kernels = gradients(case, dev(case["Ind"]), X, dev(case["Y"]))
    assert kernels.count("tiled_dw_split_kernel") == 2, kernels
    assert_close(dWg, O.gather_backward(np64(case["X"]), np64(case["Wg"]), case["Ind"].numpy(), np64(case["Y"]))[1], torch.float32, "dWg")
    assert_close(dWs, O.scatter_backward(np64(case["Y"]), np64(case["Ws"]), case["Ind"].numpy(), np64(case["dOut"]))[1], torch.float32, "dWs")


def test_values_that_have_no_three_pieces():
    """Infinities, NaN and values that round to infinity in bf16 give what the fp32 instruction gives, and stay with their results."""
    B, T, E, K, I, J = 4, 50, 3, 130, 70, 66
    case = make_case(6, B, T, E, K, I, J, torch.float32)
    X, Y = case["X"].clone(), case["Y"].clone()
    Ind = case["Ind"] % (T - 3)
    Ind[1, 0, 7], Ind[2, 1, 9], Ind[3, 2, 11] = T - 1, T - 2, T - 3     # picked once each
    X[1, T - 1, 5] = float("inf")
    X[2, T - 2, 69] = float("nan")
    X[3, T - 3, 64] = 3.4e38
    Y[3, 2, 11] *= 1e-3
    got, _, kernels = gradients(case, dev(Ind), dev(X), dev(Y))
    assert kernels.count("tiled_dw_split_kernel") == 2, kernels
    got = got.cpu().double()
    bi = torch.arange(B)[:, None, None]
    want = torch.einsum("beki,bekj->eij", X.double()[bi, Ind], Y.double())
    assert torch.equal(got.isnan(), want.isnan()) and want.isnan().sum() == J
    assert torch.equal(got.isinf(), want.isinf()) and want.isinf().sum() == J and torch.equal(got[want.isinf()], want[want.isinf()])
    big = want.abs() > 1e30
    fine = want.isfinite() & ~big
    assert (big & want.isfinite()).sum() == J and torch.allclose(got[big], want[big], rtol=1e-5)
    assert (got[fine] - want[fine]).abs().max() <= 1e-4 * want[fine].abs().max()


@pytest.mark.parametrize("x_exp, y_exp", [(-100, 0), (-120, 20), (10, -120), (-140, 40), (-60, -70), (100, -100), (112, -60), (-120, 117), (60, 40)])
def test_operands_of_any_magnitude(x_exp, y_exp):
    """Operands down to the smallest subnormal number and up to 2^120: as close to 64 bits as a rounding of each product and sum, of which
    those below 2^-126 have an absolute one of 2^-150."""
    B, T, E, K, I, J = 8, 40, 3, 65, 65, 63
    case = make_case(11, B, T, E, K, I, J, torch.float32)
    X, Y = (case["X"].double() * 2.0 ** x_exp).float(), (case["Y"].double() * 2.0 ** y_exp).float()
    dWg, _, kernels = gradients(case, dev(case["Ind"]), dev(X), dev(Y))
    assert kernels.count("tiled_dw_split_kernel") == 2, kernels
    want = O.gather_backward(np64(X), np64(case["Wg"]), case["Ind"].numpy(), np64(Y))[1]
    n = (B * K) ** 0.5
    limit = 4 * 2.0 ** -24 * n * np.sqrt((want ** 2).mean()) + 4 * 2.0 ** -150 * n
    assert np.sqrt(((np64(dWg) - want) ** 2).mean()) <= limit


def test_one_pick_is_one_rounding():
    """The weight gradient of an expert with one pick: each product rounded once, as fp32 gives it."""
    B, T, E, K, I, J = 1, 9, 640, 1, 67, 35
    case = make_case(12, B, T, E, K, I, J, torch.float32)
    dWg, dWs, kernels = gradients(case, dev(case["Ind"]), dev(case["X"]), dev(case["Y"]))
    assert kernels.count("tiled_dw_wide_kernel") == 2, kernels
    x, y, do = (t.double()[0] for t in (case["X"], case["Y"], case["dOut"]))
    token = case["Ind"][0, :, 0]
    assert torch.equal(dWg.cpu(), (x[token][:, :, None] * y[:, 0][:, None, :]).float())
    assert torch.equal(dWs.cpu(), (y[:, 0][:, :, None] * do[token][:, None, :]).float())


@pytest.mark.parametrize("I, J", [(37, 29), (70, 66), (129, 1)])
def test_what_lies_between_the_rows_does_not_count(I, J):
    """Views whose gaps hold NaN give the bits of views whose gaps hold zeros: no wavefront does its tile again for columns nobody stores."""
    B, T, E, K = 9, 21, 5, 60
    case = make_case(13, B, T, E, K, I, J, torch.float32)
    got = []
    for gap in (0.0, float("nan")):
        X = torch.full((B, T, I + 5), gap, device="cuda")
        X[..., :I] = dev(case["X"])
        dW = torch.empty(E, I, J, device="cuda")
        dims = _abi.Dims(B, T, E, K, I, J)
        n = _abi.lib().egs_workspace_bytes(_abi.OP_DW, 0, dims, _abi.F32)
        ws = torch.empty(n, dtype=torch.uint8, device="cuda")
        Y = torch.full((B * E * K * J + 64,), gap, device="cuda")[:B * E * K * J].view(B, E, K, J).copy_(dev(case["Y"]))
        Ind = dev(case["Ind"])
        with _abi.launch_log() as log:
            rc = _abi.lib().egs_dw(X.data_ptr(), Y.data_ptr(), Ind.data_ptr(), dW.data_ptr(), ws.data_ptr(), n, dims, X.stride(0), X.stride(1),
                                   _abi.F32, _abi.F32, _abi.IND_I64, 0, torch.cuda.current_stream().cuda_stream)
        assert rc == 0 and log.kernels[0] == "tiled_dw_split_kernel", (rc, log.kernels)
        got.append(dW)
    assert torch.equal(*got)
    assert_close(got[0], O.gather_backward(np64(case["X"]), np64(case["Wg"]), case["Ind"].numpy(), np64(case["Y"]))[1], torch.float32, "dW")


def test_finite_results_keep_their_bits_beside_others():
    B, T, E, K, I, J = 4, 50, 3, 130, 70, 66
    case = make_case(14, B, T, E, K, I, J, torch.float32)
    Ind, Y = dev(case["Ind"]), dev(case["Y"])
    plain = gradients(case, Ind, dev(case["X"]), Y)[0]
    X = case["X"].clone()
    X[:, :, 7], X[:, :, 40], X[:, :, 69] = float("inf"), float("nan"), 2.0 ** 113
    got, _, kernels = gradients(case, Ind, dev(X), Y)
    assert kernels.count("tiled_dw_split_kernel") == 2, kernels
    rows = [i for i in range(I) if i not in (7, 40, 69)]
    assert torch.equal(got[:, rows], plain[:, rows])
    assert not got[:, [7, 40]].isfinite().any()
    want = O.gather_backward(np64(X[:, :, 69:]), np64(case["Wg"][:, 69:]), case["Ind"].numpy(), np64(case["Y"]))[1]
    assert_close(got[:, 69:], want, torch.float32, "dW")


def test_sources_from_2_gib_on():
    """A view that spans more than 2 GiB: the fp32 instruction's kernel, in as many parts as that one takes."""
    B, T, E, K, I, J = 3, 30, 2, 200, 70, 66
    case = make_case(15, B, T, E, K, I, J, torch.float32)
    X = torch.empty(2 * (2 ** 28 + 64) + T * I, device="cuda").as_strided((B, T, I), (2 ** 28 + 64, I, 1)).copy_(case["X"])
    Y, Ind = dev(case["Y"]), dev(case["Ind"])
    dW = torch.empty(E, I, J, device="cuda")
    dims = _abi.Dims(B, T, E, K, I, J)
    n = _abi.lib().egs_workspace_bytes(_abi.OP_DW, 0, dims, _abi.F32)
    ws = torch.empty(n, dtype=torch.uint8, device="cuda")
    with _abi.launch_log() as log:
        rc = _abi.lib().egs_dw(X.data_ptr(), Y.data_ptr(), Ind.data_ptr(), dW.data_ptr(), ws.data_ptr(), n, dims, X.stride(0), X.stride(1),
                               _abi.F32, _abi.F32, _abi.IND_I64, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and log.kernels == ["tiled_dw_kernel"], (rc, log.kernels)
    assert_close(dW, O.gather_backward(np64(case["X"]), np64(case["Wg"]), case["Ind"].numpy(), np64(case["Y"]))[1], torch.float32, "dW")


@pytest.mark.parametrize("shape, kernel", [((12, 121, 52, 61, 272, 31), "tiled_dw_kernel"),         # 59 % of the 64 x 64 tiles empty
                                           ((26, 60, 30, 30, 523, 32), "tiled_dw_kernel"),
                                           ((1, 40, 640, 40, 3, 5), "tiled_dw_wide_kernel"),        # fewer than 64 picks
                                           ((8, 30, 90, 8, 66, 130), "tiled_dw_split_kernel"),      # 64 picks
                                           ((53, 97, 29, 41, 111, 75), "tiled_dw_split_kernel")], ids=lambda s: "x".join(map(str, s)) if isinstance(s, tuple) else None)
def test_where_the_split_kernel_is_taken(shape, kernel):
    case = make_case(16, *shape, torch.float32)
    dWg, _, kernels = gradients(case, dev(case["Ind"]), dev(case["X"]), dev(case["Y"]))
    assert kernels.count(kernel) == 2, kernels
    assert_close(dWg, O.gather_backward(np64(case["X"]), np64(case["Wg"]), case["Ind"].numpy(), np64(case["Y"]))[1], torch.float32, "dW")
