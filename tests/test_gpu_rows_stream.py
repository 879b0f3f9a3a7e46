"""rows_stream_kernel (csrc/egs_rows_stream.h): products of experts with few rows, whose weights stream through LDS; both weight layouts,
gathered and dense rows, fp8 weights, tails of rows and columns, picks that do not exist; against the oracle."""
import pytest
import torch

from expertscattergather_amd import workloads
from oracle import egs_oracle as O
from tests._util import assert_close, make_case, np64
from tests.test_gpu_parity import dev

pytestmark = pytest.mark.gpu

from expertscattergather_amd import _abi
from expertscattergather_amd import hip_kernels as hk

# I and J both take the parts of reduction (multiples of 64 from 384 on) and columns
SHAPES = [(1, 9, 3, 1, 384, 384),          # one row, six slabs: three in flight from the start, three more
          (2, 40, 5, 16, 448, 384),        # 32 rows: one tile
          (3, 40, 4, 11, 384, 512),        # 33 rows: two tiles, the second with one row
          (4, 50, 2, 32, 576, 392),        # 128 rows; 392 columns (and a reduction of 392, which is not for this kernel)
          (2, 33, 20, 17, 1024, 1024)]     # 34 rows: two tiles, the second with two rows


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_products_of_few_rows(shape, dtype):
    B, T, E, K, I, J = shape
    case = make_case(sum(shape), *shape, dtype, ind_dtype=torch.int16 if K == 17 else torch.int64)
    Ind = case["Ind"].clone()
    if B > 1:
        Ind[0, 0, 0], Ind[-1, -1, -1] = T, -1
    keep = ((Ind >= 0) & (Ind < T)).numpy()[..., None]
    safe = Ind.clamp(0, T - 1).to(torch.int64).numpy()
    X, Wg, Ws, Y, dOut, Id = (dev(t) for t in (case["X"], case["Wg"], case["Ws"], case["Y"], case["dOut"], Ind))
    x, wg, ws, y, do = (np64(case[k]) for k in ("X", "Wg", "Ws", "Y", "dOut"))

    def streamed(call, yes=True):
        with _abi.launch_log() as log:
            r = call()
        assert (log.kernels[0] == "rows_stream_kernel") == yes, log.kernels
        return r
    got = streamed(lambda: hk.expert_gather_forward_call(X, Wg, Id, torch.float32))
    assert_close(got, O.gather_forward(x, wg, safe) * keep, dtype, "Y")
    wide = torch.full((B, T + 1, I + 8), float("nan"), dtype=dtype, device="cuda")
    wide[:, :T, :I] = X
    assert torch.equal(streamed(lambda: hk.expert_gather_forward_call(wide[:, :T, :I], Wg, Id, torch.float32)), got)
    dY, _ = streamed(lambda: hk.expert_scatter_backward_call(Y, Ws, Id, dOut, torch.float32))
    assert_close(dY, O.gather_forward(do, ws.transpose(0, 2, 1), safe) * keep, dtype, "dY")
    out = streamed(lambda: hk.expert_scatter_forward_call(Y, Ws, Id, T, torch.float32), J % 64 == 0)
    assert_close(out, O.scatter_forward(y * keep, ws, safe, T), dtype, "out")
    dX, _ = streamed(lambda: hk.expert_gather_backward_call(X, Wg, Id, Y, torch.float32), J % 64 == 0)
    assert_close(dX, O.gather_backward(x, wg, safe, y * keep)[0], dtype, "dX")


@pytest.mark.parametrize("shape", [(2, 40, 64, 16, 448, 128), (3, 40, 57, 10, 384, 144), (1, 33, 31, 40, 512, 304), (2, 20, 130, 20, 384, 1024)], ids=lambda s: "x".join(map(str, s)))
def test_fp8_weights(shape):
    B, T, E, K, I, J = shape
    case = make_case(sum(shape), *shape, torch.bfloat16)
    Ind = case["Ind"].clone()
    Ind[0, 0, 0], Ind[-1, -1, -1] = T, -1
    Wq, scale = workloads.quantize_fp8_weights(dev(case["Wg"]))
    with _abi.launch_log() as log:
        got = hk.expert_gather_fp8w_forward(dev(case["X"]), Wq, scale, dev(Ind))
    assert log.kernels == ["rows_stream_kernel"], log.kernels
    w = np64(Wq.float()) * np64(scale)[:, None, :]
    assert_close(got, O.gather_forward(np64(case["X"]), w, Ind.clamp(0, T - 1).numpy()) * ((Ind >= 0) & (Ind < T)).numpy()[..., None], torch.bfloat16, "Y")


@pytest.mark.parametrize("act", ["none", "relu", "gelu", "silu"])
def test_bias_and_activation(act):
    B, T, E, K, I, J = 3, 40, 4, 11, 384, 136
    case = make_case(9, B, T, E, K, I, J, torch.bfloat16)
    X, Wg, Ind = dev(case["X"]), dev(case["Wg"]), dev(case["Ind"])
    bias = dev(torch.randn(E, J, generator=torch.Generator().manual_seed(1)).bfloat16()) if act == "none" else None
    Y = torch.empty(B, E, K, J, dtype=torch.bfloat16, device="cuda")
    code = {"none": 0, "relu": 1, "gelu": 2, "silu": 3}[act]
    with _abi.launch_log() as log:
        rc = _abi.lib().egs_expert_gather_act_forward(X.data_ptr(), Wg.data_ptr(), bias.data_ptr() if bias is not None else None, Ind.data_ptr(), Y.data_ptr(), None, 0,
                                                      _abi.Dims(B, T, E, K, I, J), T * I, I, _abi.BF16, _abi.IND_I64, code, torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and log.kernels == ["rows_stream_kernel"], (rc, log.kernels)
    want = torch.from_numpy(O.gather_forward(np64(case["X"]), np64(case["Wg"]), case["Ind"].numpy()))
    if bias is not None:
        want = want + bias.cpu().double()[None, :, None, :]
    want = {"none": lambda v: v, "relu": torch.relu, "gelu": torch.nn.functional.gelu, "silu": torch.nn.functional.silu}[act](want)
    assert_close(Y, want.numpy(), torch.bfloat16, act)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_scatter_with_bias(dtype):
    B, T, E, K, I, J = 3, 40, 7, 11, 136, 448
    case = make_case(10, B, T, E, K, I, J, dtype)
    Ind = case["Ind"].clone()
    Ind[0, 0, 0], Ind[-1, -1, -1] = T, -1
    bias = torch.randn(E, 1, I, generator=torch.Generator().manual_seed(2)).to(dtype)
    with _abi.launch_log() as log:
        out = hk.expert_scatter(dev(case["Y"]), dev(case["Ws"]), dev(Ind), T, "deterministic", dev(bias))
    assert log.kernels == ["rows_stream_kernel", "token_sum_kernel"], log.kernels
    keep = (Ind >= 0) & (Ind < T)
    picks = torch.zeros(B * T, E, dtype=torch.float64)
    b, e, _ = keep.nonzero(as_tuple=True)
    picks.index_put_((Ind[keep] + b * T, e), torch.ones((), dtype=torch.float64), accumulate=True)
    want = O.scatter_forward(np64(case["Y"]) * keep.numpy()[..., None], np64(case["Ws"]), Ind.clamp(0, T - 1).numpy(), T)
    assert_close(out, want + (picks.numpy() @ np64(bias[:, 0])).reshape(B, T, I), dtype, "out")


@pytest.mark.parametrize("rows", [20, 40])
def test_weights_past_the_caches(rows):
    """More weights than the line (128 MB), under a single row tile of 32 or 64 rows: read past the caches."""
    B, T, E, K, I, J = 1, 64, 340, rows, 1024, 512
    g = torch.Generator(device="cuda").manual_seed(2)
    X, W = (torch.randn(*s, device="cuda", generator=g).bfloat16() for s in ((B, T, I), (E, I, J)))
    Ind = torch.randint(0, T, (B, E, K), device="cuda", generator=g)
    with _abi.launch_log() as log:
        Y = hk.expert_gather_forward_call(X, W, Ind, torch.float32)
    assert log.kernels == ["rows_stream_kernel"], log.kernels
    want = torch.stack([X[0, Ind[0, e]].float() @ W[e].float() for e in range(E)])
    assert (Y[0].float() - want).abs().max() <= 2 * 2.0 ** -8 * want.abs().max()


@pytest.mark.parametrize("dims, streamed", [((1, 200, 114, 128, 1984, 256), False),         # four row tiles of many weights
                                            ((1, 64, 251, 26, 1280, 312), False),           # weight rows of no whole lines, more than a round
                                            ((2, 64, 88, 58, 1408, 128), True),             # one round
                                            ((1, 64, 206, 30, 704, 256), True)], ids=lambda d: "x".join(map(str, d)) if isinstance(d, tuple) else None)
def test_where_weights_stream(dims, streamed):
    B, T, E, K, I, J = dims
    g = torch.Generator(device="cuda").manual_seed(3)
    X, W = (torch.randn(*s, device="cuda", generator=g).bfloat16() for s in ((B, T, I), (E, I, J)))
    Ind = torch.randint(0, T, (B, E, K), device="cuda", generator=g)
    with _abi.launch_log() as log:
        Y = hk.expert_gather_forward_call(X, W, Ind, torch.float32)
    assert (log.kernels == ["rows_stream_kernel"]) == streamed, log.kernels
    want = torch.stack([torch.stack([X[b, Ind[b, e]].float() @ W[e].float() for e in range(E)]) for b in range(B)])
    assert (Y.float() - want).abs().max() <= 2 * 2.0 ** -8 * want.abs().max()
