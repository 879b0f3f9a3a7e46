"""Which scatter a call takes (scatter_choose, small_token_sums_pay in csrc/egs_lib.hip): sizes on both sides of each rule, at the edges of units of 32
picks, of passes and of token groups.  The one-kernel scatter needs no workspace and stays where none is given: both ways match the oracle."""
import ctypes

import pytest
import torch

from oracle import egs_oracle as O
from tests._util import assert_close, make_case, np64
from tests.test_gpu_parity import dev

pytestmark = pytest.mark.gpu

from expertscattergather_amd import _abi
from expertscattergather_amd import hip_kernels as hk

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
EJI = 1                         # weights [E,J,I]


def case_of(shape, dtype):
    B, T, E, K, I, J = shape
    case = make_case(sum(shape), *shape, dtype)
    Ind = torch.randint(0, T, (B, E, K), generator=torch.Generator().manual_seed(K))        # with repeats
    Ind[0, 0, 0], Ind[-1, -1, -1] = T, -1               # picks that do not exist
    Y = np64(case["Y"]) * ((Ind >= 0) & (Ind < T)).numpy()[..., None]
    return case, Ind, Ind.clamp(0, T - 1).numpy(), Y


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("shape, by_rows", [
    ((2, 454, 83, 5, 160, 64), ("bf16", "f16", "f32")),     # few picks per expert
    ((9, 454, 28, 5, 96, 64), ("f32",)),                    # few batch elements, many tokens: fp32 alone
    ((40, 64, 8, 32, 64, 64), ()),                          # full units
    ((3, 33, 31, 33, 96, 64), ("f32",)),                    # 1023 picks, the second unit of one pick
    ((4, 40, 52, 40, 96, 64), ("bf16", "f16", "f32")),      # 2080 picks: passes lose
    ((39, 43, 49, 25, 96, 32), ()),                         # and win: short rows and few tokens
    ((12, 65, 110, 8, 64, 32), ("f32",)),                   # units of eight picks that a routing table does not make up for in fp32
], ids=lambda s: "x".join(map(str, s)) if s and isinstance(s[0], int) else None)
def test_with_and_without_a_workspace(shape, by_rows, dtype):
    B, T, E, K, I, J = shape
    case, Ind, safe, Y = case_of(shape, DTYPES[dtype])
    L, d, code = _abi.lib(), _abi.Dims(*shape), hk.dtype_to_type_id(DTYPES[dtype])
    Yd, Ws, Indd = dev(case["Y"]), dev(case["Ws"]), dev(Ind)
    want = O.scatter_forward(Y, np64(case["Ws"]), safe, T)
    planned = L.egs_workspace_bytes(1, 0, d, code)
    assert (planned > 0) == (dtype in by_rows), planned
    assert L.egs_workspace_bytes(1, _abi.SCATTER_COMPACT, d, code) == 0
    ws = torch.empty(2 * planned + 512, dtype=torch.uint8, device="cuda")
    # (bytes, offset): the rows with what is asked for or more, else the one kernel, which needs none
    first = {}
    for size, at in sorted({(planned, 0), (2 * planned, 0), (max(planned - 1, 0), 0), (planned, 8), (0, 0)}):
        out = torch.full((B, T, I), float("nan"), dtype=DTYPES[dtype], device="cuda")
        with _abi.launch_log() as log:
            rc = L.egs_gemm_scatter(Yd.data_ptr(), Ws.data_ptr(), Indd.data_ptr(), out.data_ptr(), ws.data_ptr() + at if size else None, size,
                                    ctypes.byref(d), code, _abi.IND_I64, EJI, 0, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, (rc, size, at, planned)
        rows = 0 < planned <= size and at == 0
        assert any(k.startswith("scatter_fused") for k in log.kernels) != rows, (size, at, log.kernels)
        assert_close(out, want, DTYPES[dtype], "out, %d bytes of workspace" % size)
        assert torch.equal(out, first.setdefault(rows, out)), (size, at)        # each way has its bits, whatever the memory
    dX, dW = hk.expert_gather_backward_call(dev(case["X"]), dev(case["Wg"]), Indd, Yd, torch.float32)
    wX, wW = O.gather_backward(np64(case["X"]), np64(case["Wg"]), safe, Y)
    assert_close(dX, wX, DTYPES[dtype], "dX")
    assert_close(dW, wW, DTYPES[dtype], "dW")


@pytest.mark.parametrize("shape, without", [
    ((1, 476, 47, 81, 56, 32), True),       # the table would be one workgroup's work
    ((9, 130, 56, 52, 32, 32), True),
    ((33, 130, 56, 52, 32, 32), False),     # a batch element more than the rule takes
    ((2, 60, 50, 40, 96, 64), False),       # more than 32 picks a token
    ((6, 70, 4, 9, 32, 64), False),
    ((1, 2100, 5, 6, 64, 32), True),        # a table for long sequences is a launch of its own
    ((2, 300, 41, 100, 64, 32), True),      # 4100 picks: few tokens
    ((2, 2100, 2150, 2, 32, 32), True),     # 4300
    ((2, 2100, 4100, 2, 32, 32), False),    # too many picks for sums without one
    ((9, 2100, 2150, 2, 32, 32), False),    # too many tokens for that many
], ids=lambda s: "x".join(map(str, s)) if isinstance(s, tuple) else str(s))
def test_sums_of_small_experts_rows(shape, without):
    case, Ind, safe, Y = case_of(shape, torch.bfloat16)
    d, code = _abi.Dims(*shape), hk.dtype_to_type_id(torch.bfloat16)
    if _abi.lib().egs_workspace_bytes(1, 0, d, code) == 0:
        pytest.skip("one kernel")
    with _abi.launch_log() as log:
        out = hk.expert_scatter_forward_call(dev(case["Y"]), dev(case["Ws"]), dev(Ind), shape[1], torch.float32)
    assert "rows_small_kernel" in log.kernels and ("token_sum_kernel" in log.kernels) == without, log.kernels
    assert_close(out, O.scatter_forward(Y, np64(case["Ws"]), safe, shape[1]), torch.bfloat16, "out")


def test_a_table_that_is_not_asked_for_is_still_taken():
    """fp32 sizes whose scatters go by rows: a caller that brings memory for a table all the same gets the same results, the table in it."""
    B, T, E, K, I, J = shape = (12, 65, 110, 8, 64, 32)
    case, Ind, safe, Y = case_of(shape, torch.float32)
    L, d, st = _abi.lib(), _abi.Dims(*shape), torch.cuda.current_stream().cuda_stream
    assert L.egs_routing_table_bytes(d, _abi.F32) == 0
    up = lambda n: (n + 255) // 256 * 256
    perm_at, nb = up(B * (T + 1) * 4), up(B * (T + 1) * 4) + up(B * E * K * 4)
    X, Wg, Ws, Yd, Indd = (dev(t) for t in (case["X"], case["Wg"], case["Ws"], case["Y"], Ind))
    table = torch.full((nb,), 0xEE, dtype=torch.uint8, device="cuda")
    Yg = torch.empty(B, E, K, J, device="cuda")
    assert L.egs_expert_gather_forward_table(X.data_ptr(), Wg.data_ptr(), Indd.data_ptr(), Yg.data_ptr(), table.data_ptr(), nb, ctypes.byref(d), T * I, I,
                                             _abi.F32, _abi.IND_I64, st) == 0
    keep = ((Ind >= 0) & (Ind < T))
    assert_close(Yg, O.gather_forward(np64(case["X"]), np64(case["Wg"]), safe) * keep.numpy()[..., None], torch.float32, "Y")
    seg = table[:perm_at].view(torch.int32)[: B * (T + 1)].reshape(B, T + 1).cpu()
    counts = torch.stack([torch.bincount(Ind[b][keep[b]], minlength=T) for b in range(B)])
    assert torch.equal(seg[:, 1:] - seg[:, :-1], counts.to(torch.int32))
    want = O.scatter_forward(Y, np64(case["Ws"]), safe, T)
    ws = torch.empty(L.egs_workspace_bytes(1, 0, d, _abi.F32), dtype=torch.uint8, device="cuda")
    for size in (ws.numel(), 0):
        out = torch.empty(B, T, I, device="cuda")
        assert L.egs_expert_scatter_bias_forward(Yd.data_ptr(), Ws.data_ptr(), None, Indd.data_ptr(), table.data_ptr(), nb, out.data_ptr(), ws.data_ptr(),
                                                 size, ctypes.byref(d), _abi.F32, _abi.IND_I64, 0, st) == 0
        assert_close(out, want, torch.float32, "out, %d bytes of workspace" % size)
