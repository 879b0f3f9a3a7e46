"""tiled_pair_kernel (csrc/egs_split_f32.h): a backward call's product and weight gradient in one launch, for every width of the product's tiles and
every kind of weight gradient, with and without splits; the bits of the two launched apart."""
import ctypes

import pytest
import torch

from oracle import egs_oracle as O
from tests._util import assert_close, make_case, np64
from tests.test_gpu_parity import dev

pytestmark = pytest.mark.gpu

from expertscattergather_amd import _abi
from expertscattergather_amd import hip_kernels as hk

OP_SCATTER, OP_DW = 1, 2


def apart(op, *args):
    """One launcher of the C ABI with a workspace of the size it asks for."""
    rc = op(*args, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, rc


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("shape", [
    (1, 9, 1, 3, 9, 11),            # one workgroup of each, a few picks
    (2, 60, 9, 70, 33, 30),         # 140 picks: 32-column tiles, splits of none
    (9, 40, 5, 130, 62, 75),        # 1170 picks: splits
    (3, 200, 40, 90, 70, 95),       # 64 and 96 columns
    (40, 30, 12, 33, 130, 79),      # fp32: 80 columns, in bf16 pieces
    (4, 50, 130, 7, 257, 129),      # many tiles of few picks
], ids=lambda s: "x".join(map(str, s)))
def test_one_launch_has_the_bits_of_two(shape, dtype):
    B, T, E, K, I, J = shape
    case = make_case(sum(shape), *shape, dtype)
    Ind = case["Ind"].clone()
    Ind[0, 0, 0], Ind[-1, -1, -1] = T, -1               # picks that do not exist
    X, Wg, Ws, Y, dOut, Ind = (dev(t) for t in (case["X"], case["Wg"], case["Ws"], case["Y"], case["dOut"], Ind))
    with _abi.launch_log() as log:
        dX, dWg = hk.expert_gather_backward_call(X, Wg, Ind, Y, torch.float32)
        dY, dWs = hk.expert_scatter_backward_call(Y, Ws, Ind, dOut, torch.float32)
    assert log.kernels.count("tiled_pair_kernel") == 2 and log.kernels.count("tiled_rows_kernel") == 2, log.kernels

    L, d, code, ind = _abi.lib(), _abi.Dims(*shape), hk.dtype_to_type_id(dtype), _abi.IND_I64
    ws = {op: torch.empty(max(256, L.egs_workspace_bytes(op, 0, d, code)), dtype=torch.uint8, device="cuda") for op in (OP_SCATTER, OP_DW)}
    want = [torch.empty_like(t) for t in (dX, dWg, dY, dWs)]
    with _abi.launch_log() as log:
        apart(L.egs_gemm_scatter, Y.data_ptr(), Wg.data_ptr(), Ind.data_ptr(), want[0].data_ptr(), ws[OP_SCATTER].data_ptr(), ws[OP_SCATTER].numel(),
              ctypes.byref(d), code, ind, 0, 0)
        apart(L.egs_dw, X.data_ptr(), Y.data_ptr(), Ind.data_ptr(), want[1].data_ptr(), ws[OP_DW].data_ptr(), ws[OP_DW].numel(), ctypes.byref(d), T * I, I,
              code, code, ind, 0)
        apart(L.egs_gather_gemm, dOut.data_ptr(), Ws.data_ptr(), Ind.data_ptr(), want[2].data_ptr(), None, ctypes.byref(d), T * I, I, code, code, ind, 1)
        apart(L.egs_dw, dOut.data_ptr(), Y.data_ptr(), Ind.data_ptr(), want[3].data_ptr(), ws[OP_DW].data_ptr(), ws[OP_DW].numel(), ctypes.byref(d), T * I, I,
              code, code, ind, 1)
    assert "tiled_pair_kernel" not in log.kernels, log.kernels
    for name, a, b in zip(("dX", "dW of the gather", "dY", "dW of the scatter"), (dX, dWg, dY, dWs), want):
        assert torch.equal(a, b), name


@pytest.mark.parametrize("shape, dtype, gather, scatter", [
    ((30, 50, 70, 70, 65, 31), torch.float32, False, True),     # one slab of 31 columns, three of 65: dX's rows written out, dY's in the loop
    ((62, 204, 58, 131, 51, 32), torch.float32, False, False),  # two slabs of 51
    ((30, 50, 64, 70, 31, 33), torch.float32, True, True),      # a weight gradient in bf16 pieces always shares
    ((60, 50, 64, 70, 31, 33), torch.bfloat16, True, True),     # half as many tiles as the line asks for
], ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v).replace("torch.", ""))
def test_large_products_of_short_reductions_stay_apart(shape, dtype, gather, scatter):
    B, T, E, K, I, J = shape
    case = make_case(sum(shape), *shape, dtype)
    X, Wg, Ws, Y, dOut, Ind = (dev(case[k]) for k in ("X", "Wg", "Ws", "Y", "dOut", "Ind"))
    with _abi.launch_log() as log:
        dX, dWg = hk.expert_gather_backward_call(X, Wg, Ind, Y, torch.float32)
    assert ("tiled_pair_kernel" in log.kernels) == gather and "tiled_rows_kernel" in log.kernels, log.kernels
    with _abi.launch_log() as log:
        dY, dWs = hk.expert_scatter_backward_call(Y, Ws, Ind, dOut, torch.float32)
    assert ("tiled_pair_kernel" in log.kernels) == scatter and "tiled_rows_kernel" in log.kernels, log.kernels
    ind = case["Ind"].numpy()
    wX, wWg = O.gather_backward(np64(case["X"]), np64(case["Wg"]), ind, np64(case["Y"]))
    wY, wWs = O.scatter_backward(np64(case["Y"]), np64(case["Ws"]), ind, np64(case["dOut"]))
    for name, got, want in (("dX", dX, wX), ("dW of the gather", dWg, wWg), ("dY", dY, wY), ("dW of the scatter", dWs, wWs)):
        assert_close(got, want, dtype, name)
