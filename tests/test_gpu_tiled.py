"""The kernels for operands of any size and alignment (csrc/egs_tiled.h, csrc/egs_token_sum.h) where they can go wrong: edges of
tiles and slabs, rows shorter than a chunk, operands of a few bytes, picks that do not exist, hot tokens; against the oracle."""
import pytest
import torch

from oracle import egs_oracle as O
from tests._util import assert_close, make_case, np64
from tests.test_gpu_parity import dev, run_all

pytestmark = pytest.mark.gpu

from expertscattergather_amd import _abi
from expertscattergather_amd import hip_kernels as hk

SHAPES = [
    (1, 2, 1, 1, 3, 1), (1, 1, 2, 2, 1, 5), (2, 3, 2, 2, 7, 2),     # operands below 16 bytes, and just above
    (3, 9, 2, 5, 5, 3),                 # rows shorter than a chunk on both sides
    (2, 40, 9, 33, 63, 65), (2, 40, 3, 32, 65, 63),                 # one element off a slab and a tile
    (4, 50, 5, 16, 520, 17),            # nine slabs, a column tile with one column in its second 16
    (2, 70, 7, 65, 129, 81),            # 130 picks per expert: two row tiles and two rows; one column past 128 and 80
    (6, 30, 11, 29, 97, 131),           # tokens picked tens of times
    (40, 33, 13, 64, 72, 100),          # 2560 picks per expert: 40 row tiles, the weight gradient in three splits
]


@pytest.mark.parametrize("mode", ["deterministic", "atomic"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_any_size_matches_the_oracle(shape, dtype, mode):
    B, T, E, K, I, J = shape
    case = make_case(300 + sum(shape), *shape, dtype, ind_dtype=torch.int16 if dtype is torch.float16 else torch.int64)
    Ind = case["Ind"].clone()
    if E * K > 40:
        g = torch.Generator().manual_seed(1)
        Ind[torch.rand(Ind.shape, generator=g) < 0.3] = T // 2      # a token with a third of the picks: shared by the workgroup
        Ind[0, 0, 0], Ind[-1, -1, -1], Ind[-1, 0, 0] = T, -1, 30000
    bad = (Ind < 0) | (Ind >= T)
    safe = Ind.clone(); safe[bad] = 0
    keep = (~bad).numpy()[..., None]
    got = run_all(dict(case, Ind=Ind), T, mode)
    X, Wg, Ws, Y, dOut = (np64(case[k]) for k in ("X", "Wg", "Ws", "Y", "dOut"))
    Yk, In = Y * keep, safe.to(torch.int64).numpy()
    dX, dWg = O.gather_backward(X, Wg, In, Yk)
    dY, dWs = O.scatter_backward(Yk, Ws, In, dOut)
    for name, ref in (("Y", O.gather_forward(X, Wg, In) * keep), ("out", O.scatter_forward(Yk, Ws, In, T)), ("dX", dX), ("dWg", dWg),
                      ("dY", dY * keep), ("dWs", dWs)):
        if mode == "atomic" and dtype is not torch.float32 and name in ("out", "dX"):     # one more rounding per pick
            assert abs(np64(got[name]) - ref).max() <= 2 ** (-6 if dtype is torch.bfloat16 else -9) * abs(ref).max() + 1e-30
        else:
            assert_close(got[name], ref, dtype, f"{name} {shape} {dtype} {mode}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("dims", [(1, 1), (3, 1), (1, 4), (1, 5), (7, 1), (1, 7), (2, 4), (8, 1), (3, 3)], ids=lambda d: "x".join(map(str, d)))
def test_experts_of_a_few_bytes(dims, dtype):
    """16-byte reads of a matrix of less than 16 bytes could not stay inside W: element by element there, by tiles from 16 on."""
    I, J = dims
    B, T, E, K = 3, 30, 5, 6
    case = make_case(40 + I + 9 * J, B, T, E, K, I, J, dtype)
    X, Wg, Ws, Y, Ind = (dev(case[k]) for k in ("X", "Wg", "Ws", "Y", "Ind"))
    with _abi.launch_log() as log:
        got = hk.expert_gather_forward_call(X, Wg, Ind, torch.float32)
        out = hk.expert_scatter_forward_call(Y, Ws, Ind, T, torch.float32)
    rows = [k for k in log.kernels if "rows" in k]
    assert rows == ["tiled_rows_kernel" if I * J * X.element_size() >= 16 else "tiny_rows_kernel"] * 2, log.kernels
    assert_close(got, O.gather_forward(np64(case["X"]), np64(case["Wg"]), case["Ind"].numpy()), dtype, "Y")
    assert_close(out, O.scatter_forward(np64(case["Y"]), np64(case["Ws"]), case["Ind"].numpy(), T), dtype, "out")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("shape", [(1, 3, 2, 600, 1, 5), (1, 2, 3, 2100, 1, 9), (1, 0, 2, 2100, 3, 5)], ids=lambda s: "x".join(map(str, s)))
def test_weight_gradient_of_sources_below_16_bytes_with_many_picks(shape, dtype):
    """More picks than one workgroup usually takes, of a source that holds no 16-byte chunk (or nothing): tiny_dw_kernel sums them all."""
    B, T, E, K, I, J = shape
    case = make_case(3, B, max(T, 1), E, K, I, J, dtype)
    X, Y, Ind = dev(case["X"][:, :T]), dev(case["Y"]), dev(case["Ind"])
    dW = torch.full((E, I, J), float("nan"), dtype=dtype, device="cuda")
    dims = _abi.Dims(B, T, E, K, I, J)
    code, n = hk.dtype_to_type_id(dtype), _abi.lib().egs_workspace_bytes(_abi.OP_DW, 0, dims, hk.dtype_to_type_id(dtype))
    ws = torch.full((max(n, 256) // 4,), float("nan"), device="cuda")
    with _abi.launch_log() as log:
        rc = _abi.lib().egs_dw(X.data_ptr() or Y.data_ptr(), Y.data_ptr(), Ind.data_ptr(), dW.data_ptr(), ws.data_ptr(), n, dims, T * I, I, code, code,
                               _abi.IND_I64, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and log.kernels == ["tiny_dw_kernel"], (rc, log.kernels)
    want = O.gather_backward(np64(case["X"]), np64(case["Wg"]), case["Ind"].numpy(), np64(case["Y"]))[1] if T else torch.zeros(E, I, J).double().numpy()
    assert_close(dW, want, dtype, "dW")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_odd_views_and_values_that_are_not_finite_stay_where_they_are(dtype):
    """X as a view with odd strides that ends at its storage's last element, W and Y off the 16-byte grid (through the C ABI's
    Python route they would be copied); a NaN row reaches only its own picks although row tails are read 16 bytes at a time."""
    B, T, E, K, I, J = 3, 21, 4, 9, 37, 29
    case = make_case(77, B, T, E, K, I, J, dtype)
    X = case["X"].clone()
    X[1, 5] = float("nan")
    wide = torch.full((B * T * 41,), float("nan"), dtype=dtype, device="cuda")
    Xv = wide[wide.numel() - ((B - 1) * T * 41 + (T - 1) * 41 + I):].as_strided((B, T, I), (T * 41, 41, 1))
    Xv.copy_(X)
    W, Ind = dev(case["Wg"]), dev(case["Ind"])
    Wo = torch.empty(W.numel() + 1, dtype=dtype, device="cuda")[1:].view(W.shape).copy_(W)
    Yo = torch.empty(B * E * K * J + 1, dtype=dtype, device="cuda")[1:].view(B, E, K, J)
    rc = _abi.lib().egs_expert_gather_forward(Xv.data_ptr(), Wo.data_ptr(), Ind.data_ptr(), Yo.data_ptr(), _abi.Dims(B, T, E, K, I, J),
                                              T * 41, 41, hk.dtype_to_type_id(dtype), _abi.IND_I64, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    hit = ((case["Ind"] == 5) & (torch.arange(B) == 1)[:, None, None])[..., None]
    assert torch.isnan(Yo.cpu().float()).eq(hit.expand(B, E, K, J)).all()
    want = O.gather_forward(np64(case["X"]), np64(case["Wg"]), case["Ind"].numpy())
    assert_close(torch.where(hit, torch.from_numpy(want).to(dtype), Yo.cpu()), want, dtype, "Y")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("shape, split32", [((1, 20, 70, 4, 200, 150), False), ((5, 60, 45, 43, 140, 135), True), ((1, 30, 130, 17, 128, 128), False),
                                            ((3, 9, 300, 11, 5, 63), False), ((3, 9, 300, 22, 5, 63), True), ((3, 30, 11, 41, 67, 131), False), ((2, 40, 20, 64, 129, 65), False),
                                            ((1, 20, 9, 3, 35, 29), False)], ids=lambda s: "x".join(map(str, s)) if isinstance(s, tuple) else None)
def test_weight_gradient_of_experts_with_few_picks(shape, split32, dtype):
    """tiled_dw_wide_kernel, in fp32 from 64 picks on with many slabs in all tiled_dw_split_kernel: one slab, several, a part of one; both output layouts;
    picks that do not exist do not count, whatever their rows hold."""
    B, T, E, K, I, J = shape
    case = make_case(sum(shape), *shape, dtype)
    Ind, Y = case["Ind"].clone(), case["Y"].clone()
    Ind[0, 0, 0], Ind[-1, -1, -1] = T, -1
    Y[0, 0, 0] = Y[-1, -1, -1] = float("nan")
    with _abi.launch_log() as log:
        _, dWg = hk.expert_gather_backward_call(dev(case["X"]), dev(case["Wg"]), dev(Ind), dev(Y), dtype)
        _, dWs = hk.expert_scatter_backward_call(dev(Y), dev(case["Ws"]), dev(Ind), dev(case["dOut"]), dtype)
    assert log.kernels.count("tiled_dw_split_kernel" if split32 and dtype is torch.float32 else "tiled_dw_wide_kernel") == 2, log.kernels
    safe = Ind.clamp(0, T - 1).numpy()
    Yk = np64(Y)
    Yk[0, 0, 0] = Yk[-1, -1, -1] = 0
    assert_close(dWg, O.gather_backward(np64(case["X"]), np64(case["Wg"]), safe, Yk)[1], dtype, "dWg")
    assert_close(dWs, O.scatter_backward(Yk, np64(case["Ws"]), safe, np64(case["dOut"]))[1], dtype, "dWs")


@pytest.mark.parametrize("dims, sums", [((6, 200, 16, 64, 256, 192), ["rows_gemm_dl_kernel", "segment_sum_kernel"]),     # the table rides along
                                        ((6, 200, 16, 64, 256, 121), ["tiled_rows_kernel", "token_sum_kernel"]),         # it would be a launch
                                        ((6, 200, 33, 125, 256, 121), ["tiled_rows_kernel", "csr_count_kernel", "segment_sum_kernel"]),  # 4125 picks
                                        ((6, 200, 17, 241, 128, 121), ["tiled_rows_kernel", "token_sum_kernel"]),        # 4097 of short rows
                                        ((20, 120, 7, 500, 844, 25), ["tiled_rows_kernel", "csr_count_kernel", "segment_sum_kernel", "tiled_rows_kernel",
                                                                      "segment_sum_kernel"]),                            # two batch groups
                                        ((20, 120, 8, 500, 801, 24), ["tiled_rows_kernel", "token_sum_kernel"] * 2)],    # of odd rows
                         ids=["rides", "few", "many", "many-short", "groups", "groups-odd"])
def test_which_sums_follow_the_product_rows(dims, sums):
    B, T, E, K, I, J = dims
    case = make_case(sum(dims), *dims, torch.bfloat16)
    with _abi.launch_log() as log:
        out = hk.expert_scatter_forward_call(dev(case["Y"]), dev(case["Ws"]), dev(case["Ind"]), T, torch.float32)
    assert log.kernels == sums, log.kernels
    assert_close(out, O.scatter_forward(np64(case["Y"]), np64(case["Ws"]), case["Ind"].numpy(), T), torch.bfloat16, "out")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("dims, tiles", [((10, 150, 64, 100, 248, 248), "both"),      # 256 x 256, the last row tile 232 rows, the last slab 56 deep
                                         ((11, 150, 63, 93, 232, 504), "both"),       # 1023 picks; one expert short of eight per XCD
                                         ((10, 150, 32, 100, 40, 248), "gather"),     # 128 x 128, less than one slab
                                         ((10, 150, 32, 100, 248, 8), "scatter"),     # one chunk of reduction
                                         ((8, 150, 32, 125, 72, 256), "gather"),      # a whole slab and one chunk
                                         ((8, 150, 32, 125, 256, 120), "scatter")], ids=lambda d: "x".join(map(str, d)) if isinstance(d, tuple) else d)
def test_large_products_off_the_direct_to_lds_loads(dims, tiles, dtype):
    """rows_gemm_kernel with partial tiles and slabs, both weight layouts, both result types, picks that do not exist."""
    B, T, E, K, I, J = dims
    case = make_case(sum(dims), *dims, dtype)
    Ind = case["Ind"].clone()
    Ind[0, 0, 0], Ind[-1, -1, -1], Ind[1, 2, 3] = T, -1, -30000
    keep = ((Ind >= 0) & (Ind < T)).numpy()[..., None]
    safe = Ind.clamp(0, T - 1).numpy()
    X, Wg, Ws, Y, dOut, Id = (dev(t) for t in (case["X"], case["Wg"], case["Ws"], case["Y"], case["dOut"], Ind))
    x, wg, ws, y, do = (np64(case[k]) for k in ("X", "Wg", "Ws", "Y", "dOut"))

    def launch(call, runs):
        with _abi.launch_log() as log:
            r = call()
        assert (log.kernels[0] == "rows_gemm_kernel") == runs, log.kernels
        return r
    got = launch(lambda: hk.expert_gather_forward_call(X, Wg, Id, torch.float32), tiles != "scatter")
    assert_close(got, O.gather_forward(x, wg, safe) * keep, dtype, "Y")
    wide = torch.full((B, T + 1, I + 8), float("nan"), dtype=dtype, device="cuda")
    wide[:, :T, :I] = X                                                          # a view with strides of its own, other index types
    assert torch.equal(launch(lambda: hk.expert_gather_forward_call(wide[:, :T, :I], Wg, Id.int(), torch.float32), tiles != "scatter"), got)
    dY, _ = launch(lambda: hk.expert_scatter_backward_call(Y, Ws, Id, dOut, torch.float32), tiles != "scatter")
    assert_close(dY, O.gather_forward(do, ws.transpose(0, 2, 1), safe) * keep, dtype, "dY")
    want = O.scatter_forward(y * keep, ws, safe, T)
    for mode in ("deterministic", "atomic"):
        with hk.scatter_mode_scope(mode):
            out = launch(lambda: hk.expert_scatter_forward_call(Y, Ws, Id, T, torch.float32), tiles != "gather")
            dX, _ = launch(lambda: hk.expert_gather_backward_call(X, Ws.transpose(1, 2).contiguous(), Id, Y, torch.float32), tiles != "gather")
        for name, r in (("out", out), ("dX", dX)):
            if mode == "atomic":        # one more rounding per pick
                assert abs(np64(r) - want).max() <= 2 ** (-6 if dtype is torch.bfloat16 else -9) * abs(want).max(), name
            else:
                assert_close(r, want, dtype, name)
