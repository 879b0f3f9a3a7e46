"""rows_atomic_f32_kernel (csrc/egs_rows_gemm.h) in both tile sizes: ragged rows, columns and reductions, hot tokens inside a tile, more of
them than there are partial sums, picks that do not exist; against the oracle."""
import pytest
import torch

from expertscattergather_amd import _abi
from expertscattergather_amd import hip_kernels as hk
from oracle import egs_oracle as O
from tests._util import assert_close, make_case, np64
from tests.test_gpu_parity import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [5, 40, 5000], ids=["hot", "many_pairs", "spread"])
@pytest.mark.parametrize("shape", [
    (1, 5100, 9, 64, 65, 150),          # one full 64-row tile, a second column tile of one
    (5, 5100, 3, 13, 63, 7),            # a tile of 65 rows, one column short of a tile, less than a slab
    (2, 5100, 90, 65, 260, 1030),       # 540 tiles of 128 x 128: a second row tile of two, a third column tile of four, a last slab of six
], ids=lambda s: "x".join(map(str, s)))
def test_atomic_tiles_match_the_oracle(shape, tokens):
    B, T, E, K, I, J = shape
    case = make_case(sum(shape), *shape, torch.float32)
    Ind = torch.randint(0, tokens, (B, E, K), generator=torch.Generator().manual_seed(7))
    Ind[0, 0, 0], Ind[-1, -1, -1] = T, -1
    keep = ((Ind >= 0) & (Ind < T)).numpy()[..., None]
    safe = Ind.clamp(0, T - 1).numpy()
    Y, Ws, Wg = (np64(case[k]) for k in ("Y", "Ws", "Wg"))
    with _abi.launch_log() as log, torch.no_grad(), hk.scatter_mode_scope("atomic"):
        out = hk.expert_scatter_forward_call(dev(case["Y"]), dev(case["Ws"]), dev(Ind), T, torch.float32)
        dX, _ = hk.expert_gather_backward_call(dev(case["X"]), dev(case["Wg"]), dev(Ind), dev(case["Y"]), torch.float32)
    assert log.kernels.count("rows_atomic_f32_kernel") == 2, log.kernels
    assert_close(out, O.scatter_forward(Y * keep, Ws, safe, T), torch.float32, "out")
    assert_close(dX, O.gather_backward(np64(case["X"]), Wg, safe, Y * keep)[0], torch.float32, "dX")
