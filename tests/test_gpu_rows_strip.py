"""rows_strip_kernel (csrc/egs_rows_strip.h): ragged last slabs, rows and columns, reductions shorter than a slab, picks that do not exist,
rows apart, both weight layouts, fp32 and 16-bit results, bias and activation; against the oracle and, bit for bit, the general kernel."""
import pytest
import torch

from oracle import egs_oracle as O
from tests._util import assert_close, make_case, np64
from tests.test_gpu_parity import dev

pytestmark = pytest.mark.gpu

from expertscattergather_amd import _abi
from expertscattergather_amd import hip_kernels as hk


def in_general(run):
    """With the general kernels (remembered workspace sizes belong to the other ones)."""
    def switch(on):
        _abi.lib().egs_testing_force_generic(on)
        hk._ws_sizes.clear()
        hk._table_sizes.clear()
    switch(1)
    try:
        return run()
    finally:
        switch(0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("shape", [
    (1, 300, 40, 250, 72, 120),     # two row tiles, two slabs, the second of eight elements
    (7, 600, 20, 54, 392, 136),     # three tiles of rows, ragged; three of columns, the last of eight; seven slabs
    (3, 900, 24, 90, 8, 232),       # a reduction of eight elements
    (5, 700, 70, 50, 136, 56),      # columns that fill no tile
], ids=lambda s: "x".join(map(str, s)))
def test_strips_match_the_oracle_and_the_general_kernel(shape, dtype):
    B, T, E, K, I, J = shape
    case = make_case(sum(shape), *shape, dtype)
    Ind = case["Ind"].clone()
    Ind[0, 0, 0], Ind[-1, -1, -1] = T, -1               # picks that do not exist
    keep = ((Ind >= 0) & (Ind < T)).numpy()[..., None]
    safe = Ind.clamp(0, T - 1).numpy()
    X = torch.full((B, T + 3, I + 8), float("nan"), dtype=dtype)       # rows apart, NaN between them
    X[:, :T, :I] = case["X"]
    X = dev(X)[:, :T, :I]

    def run():
        with _abi.launch_log() as log:
            Y = hk.expert_gather_forward_call(X, dev(case["Wg"]), dev(Ind), torch.float32)
            out = hk.expert_scatter_forward_call(dev(case["Y"]), dev(case["Ws"]), dev(Ind), T, torch.float32)
            dX, _ = hk.expert_gather_backward_call(X, dev(case["Wg"]), dev(Ind), dev(case["Y"]), torch.float32)
            dY, _ = hk.expert_scatter_backward_call(dev(case["Y"]), dev(case["Ws"]), dev(Ind), dev(case["dOut"]), torch.float32)
        return (Y, out, dX, dY), log.kernels

    got, kernels = run()
    assert "rows_strip_kernel" in kernels, kernels
    plain, kernels = in_general(run)
    assert "rows_strip_kernel" not in kernels and "tiled_rows_kernel" in kernels, kernels
    Yk = np64(case["Y"]) * keep
    want = (O.gather_forward(np64(case["X"]), np64(case["Wg"]), safe) * keep, O.scatter_forward(Yk, np64(case["Ws"]), safe, T),
            O.gather_backward(np64(case["X"]), np64(case["Wg"]), safe, Yk)[0], O.scatter_backward(Yk, np64(case["Ws"]), safe, np64(case["dOut"]))[0] * keep)
    for name, g, p, w in zip(("Y", "out", "dX", "dY"), got, plain, want):
        assert_close(g, w, dtype, name)
        assert torch.equal(g, p), name


@pytest.mark.parametrize("act", ["none", "relu", "gelu", "silu"])
def test_bias_and_activation(act):
    B, T, E, K, I, J = 3, 400, 30, 70, 200, 120
    case = make_case(9, B, T, E, K, I, J, torch.bfloat16)
    X, Wg, Ind = dev(case["X"]), dev(case["Wg"]), dev(case["Ind"])
    bias = dev(torch.randn(E, J, generator=torch.Generator().manual_seed(1)).bfloat16()) if act == "none" else None
    code = {"none": 0, "relu": 1, "gelu": 2, "silu": 3}[act]

    def run():
        Y = torch.empty(B, E, K, J, dtype=torch.bfloat16, device="cuda")
        with _abi.launch_log() as log:
            rc = _abi.lib().egs_expert_gather_act_forward(X.data_ptr(), Wg.data_ptr(), bias.data_ptr() if bias is not None else None, Ind.data_ptr(), Y.data_ptr(), None, 0,
                                                          _abi.Dims(B, T, E, K, I, J), T * I, I, _abi.BF16, _abi.IND_I64, code, torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        return Y, log.kernels

    got, kernels = run()
    assert kernels == ["rows_strip_kernel"], kernels
    plain, kernels = in_general(run)
    assert kernels == ["tiled_rows_kernel"], kernels
    assert torch.equal(got, plain)
    if act in ("none", "relu"):
        want = O.gather_forward(np64(case["X"]), np64(case["Wg"]), case["Ind"].numpy())
        want = want + np64(bias)[None, :, None, :] if act == "none" else want.clip(0)
        assert_close(got, want, torch.bfloat16, "Y")


@pytest.mark.parametrize("mode", ["deterministic", "atomic"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_scatter_with_bias(dtype, mode):
    """The rows come with their bias, in fp32 or (atomic mode) in the element type: the general kernel's bits."""
    B, T, E, K, I, J = 3, 400, 30, 70, 120, 200
    case = make_case(10, B, T, E, K, I, J, dtype)
    Ind = case["Ind"].clone()
    Ind[0, 0, 0], Ind[-1, -1, -1] = T, -1
    bias = torch.randn(E, 1, I, generator=torch.Generator().manual_seed(2)).to(dtype)
    Y, Ws, Id, bd = (dev(t) for t in (case["Y"], case["Ws"], Ind, bias))

    def run():
        with _abi.launch_log() as log:
            out = hk.expert_scatter(Y, Ws, Id, T, mode, bd)
        return out, log.kernels

    got, kernels = run()
    assert kernels == ["rows_strip_kernel", "token_sum_kernel"], kernels
    plain, kernels = in_general(run)
    assert kernels == ["tiled_rows_kernel", "token_sum_kernel"], kernels
    assert torch.equal(got, plain)
    if mode == "deterministic":
        keep = (Ind >= 0) & (Ind < T)
        picks = torch.zeros(B * T, E, dtype=torch.float64)
        b, e, _ = keep.nonzero(as_tuple=True)
        picks.index_put_((Ind[keep] + b * T, e), torch.ones((), dtype=torch.float64), accumulate=True)
        want = O.scatter_forward(np64(case["Y"]) * keep.numpy()[..., None], np64(case["Ws"]), Ind.clamp(0, T - 1).numpy(), T)
        assert_close(got, want + (picks.numpy() @ np64(bias[:, 0])).reshape(B, T, I), dtype, "out")


@pytest.mark.parametrize("dims, strips", [((6, 90, 8, 78, 160, 128), False),        # 58 full tiles
                                          ((10, 90, 30, 25, 144, 96), True),        # 88
                                          ((16, 120, 103, 120, 160, 32), False),    # 1545 half empty strips of a short reduction
                                          ((16, 120, 103, 120, 416, 32), True),
                                          ((2, 120, 150, 12, 456, 1024), False)], ids=lambda d: "x".join(map(str, d)) if isinstance(d, tuple) else None)
def test_where_strips_are_taken(dims, strips):
    case = make_case(11, *dims, torch.bfloat16)
    with _abi.launch_log() as log:
        Y = hk.expert_gather_forward_call(dev(case["X"]), dev(case["Wg"]), dev(case["Ind"]), torch.float32)
    assert log.kernels == ["rows_strip_kernel" if strips else "tiled_rows_kernel"], log.kernels
    assert_close(Y, O.gather_forward(np64(case["X"]), np64(case["Wg"]), case["Ind"].numpy()), torch.bfloat16, "Y")
