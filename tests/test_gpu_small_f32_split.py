"""rows_small_f32_kernel (csrc/egs_small_f32.h), whose products are taken in three bf16 pieces: every width and reduction length, rows that
fill no tile, and values that have no such pieces; against the oracle."""
import numpy as np
import pytest
import torch

from oracle import egs_oracle as O
from tests._util import assert_close, make_case, np64
from tests.test_gpu_parity import dev

pytestmark = pytest.mark.gpu

from expertscattergather_amd import _abi
from expertscattergather_amd import hip_kernels as hk


def products(case, Ind, X, dOut):
    """Y of the gather (weights [E,I,J]) and dY of the scatter (weights [E,J,I])."""
    with _abi.launch_log() as log:
        Y = hk.expert_gather_forward_call(X, dev(case["Wg"]), Ind, torch.float32)
        dY, _ = hk.expert_scatter_backward_call(dev(case["Y"]), dev(case["Ws"]), Ind, dOut, torch.float32)
    assert log.kernels.count("rows_small_f32_kernel") == 2, log.kernels
    return Y, dY


@pytest.mark.parametrize("J", [16, 32, 48, 64])
@pytest.mark.parametrize("I", [32, 64, 128])
def test_products_match_the_oracle(I, J):
    B, T, E, K = 9, 50, 17, 30                          # 270 picks: a second workgroup with one wavefront of 14
    case = make_case(I + J, B, T, E, K, I, J, torch.float32)
    Ind = case["Ind"].clone()
    Ind[0, 0, 0], Ind[-1, -1, -1] = T, -1               # picks that do not exist
    keep = ((Ind >= 0) & (Ind < T)).numpy()[..., None]
    safe = Ind.clamp(0, T - 1).numpy()
    Y, dY = products(case, dev(Ind), dev(case["X"]), dev(case["dOut"]))
    for got, want, what in ((Y, O.gather_forward(np64(case["X"]), np64(case["Wg"]), safe) * keep, "Y"),
                            (dY, O.scatter_backward(np64(case["Y"]) * keep, np64(case["Ws"]), safe, np64(case["dOut"]))[0] * keep, "dY")):
        assert_close(got, want, torch.float32, what)
        # a rounding per product would be 2^-24 sqrt(I) of the result: no worse than four times that
        assert np.sqrt(((np64(got) - want) ** 2).mean()) <= 4 * 2.0 ** -24 * I ** 0.5 * np.sqrt((want ** 2).mean()), what


def test_values_that_have_no_three_pieces():
    B, T, E, K, I, J = 8, 40, 16, 32, 64, 64
    case = make_case(3, B, T, E, K, I, J, torch.float32)
    X, W = case["X"].clone(), case["Wg"]
    Ind = case["Ind"] % (T - 3)
    Ind[1, 0, 7], Ind[2, 1, 9], Ind[3, 2, 11] = T - 1, T - 2, T - 3     # picked once each
    X[1, T - 1, 5] = float("-inf")
    X[2, T - 2, 63] = float("nan")
    X[3, T - 3, 32] = 3.4e38                            # infinity in bf16
    Y, _ = products(case, dev(Ind), dev(X), dev(case["dOut"]))
    got = Y.cpu().double()
    bi = torch.arange(B)[:, None, None]
    want = torch.einsum("beki,eij->bekj", X.double()[bi, Ind], W.double())
    assert torch.equal(got.isnan(), want.isnan()) and want.isnan().sum() == J
    assert torch.equal(got.isinf(), want.isinf()) and want.isinf().sum() == J and torch.equal(got[want.isinf()], want[want.isinf()])
    big = want.isfinite() & (want.abs() > 1e30)
    assert big.sum() == J and torch.allclose(got[big], want[big], rtol=1e-5)
    fine = want.isfinite() & ~big
    assert (got[fine] - want[fine]).abs().max() <= 1e-4 * want[fine].abs().max()


@pytest.mark.parametrize("x_exp, w_exp", [(-100, 0), (-120, 20), (10, -120), (-140, 40), (-60, -70), (100, -100), (112, -60), (-120, 117), (60, 40)])
def test_operands_of_any_magnitude(x_exp, w_exp):
    """Operands down to the smallest subnormal number and up to 2^120: as close to 64 bits as a rounding of each product and sum, of which
    those below 2^-126 have an absolute one of 2^-150."""
    B, T, E, K, I, J = 8, 40, 16, 32, 64, 48
    case = make_case(4, B, T, E, K, I, J, torch.float32)
    X = (case["X"].double() * 2.0 ** x_exp).float()
    case["Wg"] = (case["Wg"].double() * 2.0 ** w_exp).float()
    Y, _ = products(case, dev(case["Ind"]), dev(X), dev(case["dOut"]))
    want = O.gather_forward(np64(X), np64(case["Wg"]), case["Ind"].numpy())
    limit = 4 * 2.0 ** -24 * I ** 0.5 * np.sqrt((want ** 2).mean()) + 4 * 2.0 ** -150 * I ** 0.5
    assert np.sqrt(((np64(Y) - want) ** 2).mean()) <= limit


def test_picks_that_do_not_exist_do_not_count_as_results():
    """Picks out of range give zeros whatever the first token's row holds, and the picks beside them keep their bits."""
    B, T, E, K, I, J = 4, 40, 16, 32, 64, 64
    case = make_case(5, B, T, E, K, I, J, torch.float32)
    Ind = case["Ind"].clamp(min=1)
    Ind[:, :, 3], Ind[:, :, 20] = T, -1
    got = []
    for first in (0.0, float("nan")):
        X = case["X"].clone()
        X[:, 0] = first
        got.append(products(case, dev(Ind), dev(X), dev(case["dOut"]))[0])
    assert torch.equal(*got) and got[0][:, :, [3, 20]].eq(0).all()


def test_finite_results_keep_their_bits_beside_others():
    B, T, E, K, I, J = 4, 40, 16, 32, 128, 64
    case = make_case(6, B, T, E, K, I, J, torch.float32)
    Ind, dOut = dev(case["Ind"]), dev(case["dOut"])
    plain = products(case, Ind, dev(case["X"]), dOut)[0]
    W = case["Wg"].clone()
    W[:, 5, 7], W[:, 6, 40], W[:, 7, 63] = float("inf"), float("nan"), 2.0 ** 113
    got = products(dict(case, Wg=W), Ind, dev(case["X"]), dOut)[0]
    columns = [j for j in range(J) if j not in (7, 40, 63)]
    assert torch.equal(got[..., columns], plain[..., columns])
    assert not got[..., [7, 40]].isfinite().any()
    want = O.gather_forward(np64(case["X"]), np64(W[:, :, 63:]), case["Ind"].numpy())
    assert_close(got[..., 63:], want, torch.float32, "Y")
