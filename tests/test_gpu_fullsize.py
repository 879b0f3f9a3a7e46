"""Full-size runs of the benchmark configurations on the GPU.

C1/C2 are compared element by element with the oracle.  C3, C4 and C5 are too large for the
float64 oracle as a whole, so they are checked (a) against the oracle on slices that are cheap to
recompute (some (b,e) blocks of the gather, one batch element of the scatter, some experts of
dW) and (b) through size-independent properties: exact linearity under scaling by 2,
adjointness of gather and scatter, bitwise repeatability of the deterministic mode, agreement
of the two scatter modes, rows nobody picks being exactly zero."""
import numpy as np
import pytest
import torch

from oracle import egs_oracle as O
from tests._util import assert_close, np64

pytestmark = pytest.mark.gpu

from expertscattergather_amd import _abi, hip_kernels as hk, workloads as wl

hk.create_kernels()
DEV = "cuda"


def gpu_inputs(name):
    cfg = wl.CONFIGS[name]
    inp = wl.make_inputs(cfg)
    return cfg, inp, {k: v.to(DEV) for k, v in inp.items()}


def test_c1_fp32_forward_matches_oracle():
    cfg, inp, g = gpu_inputs("C1")
    B, T, E, K, I, J = cfg.dims
    Y = hk.expert_gather_forward_call(g["X"], g["Wg"], g["Ind"], torch.float32)
    out = hk.expert_scatter_forward_call(Y, g["Ws"], g["Ind"], T, torch.float32)
    Indn = inp["Ind"].numpy()
    assert_close(Y, O.gather_forward(np64(inp["X"]), np64(inp["Wg"]), Indn), torch.float32, "C1 Y")
    assert_close(out, O.scatter_forward(np64(Y), np64(inp["Ws"]), Indn, T), torch.float32, "C1 out")


@pytest.mark.parametrize("mode", ["deterministic", "atomic"])
def test_c2_bf16_chain_matches_oracle(mode):
    cfg, inp, g = gpu_inputs("C2")
    B, T, E, K, I, J = cfg.dims
    hk.set_scatter_mode(mode)
    try:
        Y = hk.expert_gather_forward_call(g["X"], g["Wg"], g["Ind"], torch.float32)
        out = hk.expert_scatter_forward_call(Y, g["Ws"], g["Ind"], T, torch.float32)
        dY, dWs = hk.expert_scatter_backward_call(Y, g["Ws"], g["Ind"], g["dOut"], torch.float32)
        dX, dWg = hk.expert_gather_backward_call(g["X"], g["Wg"], g["Ind"], dY, torch.float32)
        torch.cuda.synchronize()
    finally:
        hk.set_scatter_mode("deterministic")
    Indn = inp["Ind"].numpy()
    Xn, Wgn, Wsn, dOn = (np64(inp[k]) for k in ("X", "Wg", "Ws", "dOut"))
    assert_close(Y, O.gather_forward(Xn, Wgn, Indn), torch.bfloat16, "C2 Y")
    assert_close(out, O.scatter_forward(np64(Y), Wsn, Indn, T), torch.bfloat16, "C2 out")
    dYo, dWso = O.scatter_backward(np64(Y), Wsn, Indn, dOn)
    assert_close(dY, dYo, torch.bfloat16, "C2 dY"); assert_close(dWs, dWso, torch.bfloat16, "C2 dWs")
    dXo, dWgo = O.gather_backward(Xn, Wgn, Indn, np64(dY))
    assert_close(dX, dXo, torch.bfloat16, "C2 dX"); assert_close(dWg, dWgo, torch.bfloat16, "C2 dWg")


def check_large(name, modes):
    cfg, inp, g = gpu_inputs(name)
    B, T, E, K, I, J = cfg.dims
    X, Wg, Ws, dOut, Ind = (g[k] for k in ("X", "Wg", "Ws", "dOut", "Ind"))
    Indn = inp["Ind"].numpy()
    rng = np.random.default_rng(0)

    # ---- gather: slices against the oracle, exact linearity under scaling by 2
    Y = hk.expert_gather_forward_call(X, Wg, Ind, torch.float32)
    for b, e in zip(rng.integers(0, B, 4), rng.integers(0, E, 4)):
        ref = np64(inp["X"][b])[Indn[b, e]] @ np64(inp["Wg"][e])
        assert_close(Y[b, e], ref, cfg.dtype, f"{name} Y[{b},{e}]")
    assert torch.equal(hk.expert_gather_forward_call(2 * X, Wg, Ind, torch.float32), 2 * Y)

    # ---- scatter: one batch element against the oracle, modes agree, unpicked rows are zero
    outs = {}
    for mode in modes:
        hk.set_scatter_mode(mode)
        try:
            outs[mode] = hk.expert_scatter_forward_call(Y, Ws, Ind, T, torch.float32)
            if mode == "deterministic":
                assert torch.equal(outs[mode], hk.expert_scatter_forward_call(Y, Ws, Ind, T, torch.float32))
        finally:
            hk.set_scatter_mode("deterministic")
    b = int(rng.integers(0, B))
    ref = O.scatter_forward(np64(Y[b:b + 1]), np64(inp["Ws"]), Indn[b:b + 1], T, acc=np.float64)
    picked = torch.zeros(T, dtype=torch.bool); picked[inp["Ind"][b].reshape(-1)] = True
    for mode, out in outs.items():
        assert_close(out[b:b + 1], ref, cfg.dtype, f"{name} out[{b}] {mode}")
        assert (out[b].cpu()[~picked] == 0).all()
    out = outs[modes[0]]

    # ---- adjointness: <gather(X), G> = <X, scatter_with_Wg(G)>  (fp32 sums of bf16 products)
    G = torch.randn(B, E, K, J, device=DEV, generator=torch.Generator(DEV).manual_seed(3)).to(cfg.dtype)
    dXg, dWg = hk.expert_gather_backward_call(X, Wg, Ind, G, torch.float32)
    lhs = (Y.double() * G.double()).sum().item(); rhs = (X.double() * dXg.double()).sum().item()
    scale = (Y.double().abs() * G.double().abs()).sum().item()
    assert abs(lhs - rhs) <= 2e-3 * scale, (lhs, rhs, scale)

    # ---- weight gradients: a few experts against the oracle
    dYs, dWs = hk.expert_scatter_backward_call(Y, Ws, Ind, dOut, torch.float32)
    for e in rng.integers(0, E, 2):
        rows = np.concatenate([np64(inp["X"][bb])[Indn[bb, e]] for bb in range(B)])          # [B*K, I]
        assert_close(dWg[e], rows.T @ np64(G[:, e]).reshape(B * K, J), cfg.dtype, f"{name} dWg[{e}]")
        grows = np.concatenate([np64(inp["dOut"][bb])[Indn[bb, e]] for bb in range(B)])
        assert_close(dWs[e], np64(Y[:, e]).reshape(B * K, J).T @ grows, cfg.dtype, f"{name} dWs[{e}]")
    b, e = int(rng.integers(0, B)), int(rng.integers(0, E))
    assert_close(dYs[b, e], np64(inp["dOut"][b])[Indn[b, e]] @ np64(inp["Ws"][e]).T, cfg.dtype, f"{name} dY[{b},{e}]")
    assert torch.equal(dWg, hk.expert_gather_backward_call(X, Wg, Ind, G, torch.float32)[1])


def test_c3_long_sequence_bf16():
    check_large("C3", ["deterministic", "atomic"])


def test_c4_zipf_routing_both_modes():
    check_large("C4", ["deterministic", "atomic"])
    # compact mode: the configuration's scatters (forward, and dX in the gather's backward) run in one kernel each, product
    # rows and sorted picks in LDS and no workspace at all; the other modes go through product rows in the workspace
    from expertscattergather_amd import _abi
    cfg, inp, g = gpu_inputs("C4")
    B, T, E, K, I, J = cfg.dims
    d = _abi.Dims(*cfg.dims)
    ws = {m: _abi.lib().egs_workspace_bytes(_abi.OP_GEMM_SCATTER, v, d, _abi.BF16) for m, v in
          (("deterministic", 0), ("atomic", 1), ("compact", 2))}
    assert ws["compact"] == 0 and ws["deterministic"] > B * E * K * I * 4 and ws["atomic"] > B * E * K * I * 2
    Y = hk.expert_gather_forward_call(g["X"], g["Wg"], g["Ind"], torch.float32)
    outs, dXs = {}, {}
    for mode in ("deterministic", "compact"):
        with hk.scatter_mode_scope(mode), _abi.launch_log() as log:
            outs[mode] = hk.expert_scatter_forward_call(Y, g["Ws"], g["Ind"], T, torch.float32)
            dXs[mode] = hk.expert_gather_backward_call(g["X"], g["Wg"], g["Ind"], Y, torch.float32)[0]
            again = hk.expert_scatter_forward_call(Y, g["Ws"], g["Ind"], T, torch.float32)
        assert torch.equal(outs[mode], again)
        if mode == "compact":
            assert log.kernels.count("scatter_pass_kernel") == 3 and "segment_sum_kernel" not in log.kernels, log.kernels
        else:
            assert "scatter_pass_kernel" not in log.kernels, log.kernels
    # Zipf: one token takes about a quarter of a batch element's picks; both modes round a token's fp32 sum once
    counts = torch.bincount(inp["Ind"][0].reshape(-1), minlength=T)
    assert counts.max() > 0.15 * cfg.E * cfg.K
    b = 3
    Indn = inp["Ind"].numpy()
    ref = O.scatter_forward(np64(Y[b:b + 1]), np64(inp["Ws"]), Indn[b:b + 1], T, acc=np.float64)
    assert_close(outs["compact"][b:b + 1], ref, cfg.dtype, "C4 out, compact mode")
    ref = O.gather_backward(np64(inp["X"][b:b + 1]), np64(inp["Wg"]), Indn[b:b + 1], np64(Y[b:b + 1]))[0]
    assert_close(dXs["compact"][b:b + 1], ref, cfg.dtype, "C4 dX, compact mode")
    assert_close(dXs["deterministic"][b:b + 1], ref, cfg.dtype, "C4 dX, deterministic mode")


def test_scatter_cut_into_uneven_batch_groups():
    """20 batch elements of C4's shape: 336 MB of fp32 product rows, which the library processes as
    groups of 7, 7 and 6 batch elements; elements on both sides of every group boundary against the oracle."""
    cfg = wl.CONFIGS["C4"]
    _, T, E, K, I, J = cfg.dims
    B = 20
    inp = wl.make_inputs(cfg, dims=(B, T, E, K, I, J))
    Y = torch.randn(B, E, K, J, generator=torch.Generator().manual_seed(11)).to(cfg.dtype)
    out = hk.expert_scatter_forward_call(Y.to(DEV), inp["Ws"].to(DEV), inp["Ind"].to(DEV), T, torch.float32)
    assert torch.equal(out, hk.expert_scatter_forward_call(Y.to(DEV), inp["Ws"].to(DEV), inp["Ind"].to(DEV), T, torch.float32))
    Indn = inp["Ind"].numpy()
    for b in (0, 6, 7, 13, 14, 19):
        ref = O.scatter_forward(np64(Y[b:b + 1]), np64(inp["Ws"]), Indn[b:b + 1], T, acc=np.float64)
        assert_close(out[b:b + 1], ref, cfg.dtype, f"out[{b}]")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("dims, kernels", [
    ((10, 256, 128, 64, 1024, 128), ["rows_gemm_dl_kernel", "rows_gemm_dl_kernel", "rows_strip_kernel"]),       # groups of 4, 4 and 2
    ((19, 300, 37, 255, 1024, 192), ["rows_gemm_dl_kernel"] * 6 + ["rows_strip_kernel"]),                       # six of 3 and one of 1
    ((8, 256, 128, 64, 1024, 128), ["rows_gemm_dl_kernel"] * 2)], ids=["4+4+2", "6x3+1", "4+4"])
def test_bias_of_a_scatter_cut_into_batch_groups(dims, kernels, dtype):
    """A last group with fewer rows per expert than the large product kernel takes runs the one for mid-sized experts, which adds the bias to
    its rows; the other groups' bias is added afterwards.  Elements on both sides of every group boundary against the oracle."""
    B, T, E, K, I, J = dims
    gen = torch.Generator().manual_seed(sum(dims))
    Y, Ws = torch.randn(B, E, K, J, generator=gen).to(dtype), (torch.randn(E, J, I, generator=gen) / J ** 0.5).to(dtype)
    bias, Ind = torch.randn(E, 1, I, generator=gen).to(dtype), torch.randint(0, T, (B, E, K), generator=gen)
    Yd, Wd, Id, bd = (t.to(DEV) for t in (Y, Ws, Ind, bias))
    with _abi.launch_log() as log:
        out = hk.expert_scatter(Yd, Wd, Id, T, "deterministic", bd)
    assert [k for k in log.kernels if "rows" in k] == kernels, log.kernels
    G = -(-B // len(kernels))
    for b in sorted({x for g in range(0, B, G) for x in (g, min(g + G, B) - 1)}):
        ref = O.scatter_forward(np64(Y[b:b + 1]), np64(Ws), Ind[b:b + 1].numpy(), T, acc=np.float64)
        picks = torch.zeros(T, E, dtype=torch.float64).index_put_((Ind[b].reshape(-1), torch.arange(E).repeat_interleave(K)),
                                                                  torch.ones((), dtype=torch.float64), accumulate=True)
        assert_close(out[b:b + 1], ref + (picks.numpy() @ np64(bias[:, 0]))[None], dtype, f"out[{b}]")


# Numbers of experts that are not a multiple of the eight XCDs, last row tiles of 232 / 240 rows and last column tiles of 8 columns
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("dims", [
    (8, 512, 67, 61, 2056, 128),        # 269 MB of fp32 rows in one launch, which leave as whole lines past the caches; no table
    (8, 512, 67, 62, 2056, 128),        # the same with the workgroups of the routing table first in the launch
    (8, 512, 67, 61, 1032, 128),        # 135 MB: 670 tiles, a workgroup per compute unit goes from one to the next
    (8, 300, 5, 700, 1032, 192),        # 22 row tiles of each of five experts: some workgroups have one tile more, three XCDs none
    ], ids=lambda d: "x".join(map(str, d)))
def test_large_product_rows_with_ragged_tiles(dims, dtype):
    B, T, E, K, I, J = dims
    gen = torch.Generator().manual_seed(sum(dims))
    Y, Ind = torch.randn(B, E, K, J, generator=gen).to(dtype), torch.randint(0, T, (B, E, K), generator=gen)
    W = (torch.randn(E, J, I, generator=gen) / J ** 0.5).to(dtype)
    Ind[0, 0, 0], Ind[-1, -1, -1] = T, -1
    keep = ((Ind >= 0) & (Ind < T)).numpy()[..., None]
    Yd, Wd, Id = Y.to(DEV), W.to(DEV), Ind.to(DEV)
    with _abi.launch_log() as log:
        out = hk.expert_scatter_forward_call(Yd, Wd, Id, T, torch.float32)
    assert log.kernels[0] == "rows_gemm_dl_kernel" and log.kernels.count("rows_gemm_dl_kernel") == 1, log.kernels
    assert torch.equal(out, hk.expert_scatter_forward_call(Yd, Wd, Id, T, torch.float32))
    # the same products with the weights the other way round: grad_X of a gather
    dX = hk.expert_gather_backward_call(torch.zeros(B, T, I, dtype=dtype, device=DEV), Wd.transpose(1, 2).contiguous(), Id, Yd, torch.float32)[0]
    safe = Ind.clamp(0, T - 1).numpy()
    for b in (0, B - 1):
        ref = O.scatter_forward(np64(Y[b:b + 1]) * keep[b:b + 1], np64(W), safe[b:b + 1], T, acc=np.float64)
        assert_close(out[b:b + 1], ref, dtype, f"out[{b}]")
        assert_close(dX[b:b + 1], ref, dtype, f"dX[{b}]")


def test_c5_fp8_weights_forward():
    cfg = wl.CONFIGS["C5"]
    B, T, E, K, I, J = cfg.dims
    gen = torch.Generator().manual_seed(cfg.seed)
    X = torch.randn(B, T, I, generator=gen).to(torch.bfloat16)
    Ind = wl.uniform_routing(B, T, E, K, gen)
    Wq = torch.empty(E, I, J, dtype=torch.float8_e4m3fn); scale = torch.empty(E, J)
    for e0 in range(0, E, 32):                           # quantise in chunks to bound host memory
        w = torch.randn(32, I, J, generator=gen) / I ** 0.5
        Wq[e0:e0 + 32], scale[e0:e0 + 32] = wl.quantize_fp8_weights(w)
    Xg, Wqg, sg, Ig = X.to(DEV), Wq.to(DEV), scale.to(DEV), Ind.to(DEV)
    Y = hk.expert_gather_fp8w_forward(Xg, Wqg, sg, Ig)
    rng = np.random.default_rng(1)
    for b, e in zip(rng.integers(0, B, 4), rng.integers(0, E, 4)):
        W = O.dequant_fp8_weights(Wq[e:e + 1].view(torch.uint8).numpy(), scale[e:e + 1].numpy())[0]
        assert_close(Y[b, e], np64(X[b])[Ind[b, e].numpy()] @ W, torch.bfloat16, f"C5 Y[{b},{e}]")
    assert torch.equal(hk.expert_gather_fp8w_forward(2 * Xg, Wqg, sg, Ig), 2 * Y)


def test_c5_fp8_activations_forward():
    """Configuration 5 on the fp8 matrix instruction (activations quantised per row to e4m3): the row quantiser is bit-exact
    against the oracle's on a sample of rows, slices of the product match the oracle evaluated on the same quantised
    operands to bf16 output accuracy, and the result stays within 5e-2 relative RMS of the bf16-activation gather."""
    cfg = wl.CONFIGS["C5"]
    B, T, E, K, I, J = cfg.dims
    gen = torch.Generator().manual_seed(cfg.seed)
    X = torch.randn(B, T, I, generator=gen).to(torch.bfloat16)
    Ind = wl.uniform_routing(B, T, E, K, gen)
    Wq = torch.empty(E, I, J, dtype=torch.float8_e4m3fn); scale = torch.empty(E, J)
    for e0 in range(0, E, 32):
        w = torch.randn(32, I, J, generator=gen) / I ** 0.5
        Wq[e0:e0 + 32], scale[e0:e0 + 32] = wl.quantize_fp8_weights(w)
    Xg, Wqg, sg, Ig = X.to(DEV), Wq.to(DEV), scale.to(DEV), Ind.to(DEV)
    Y, Xq, xs = hk.expert_gather_fp8_forward(Xg, Wqg, sg, Ig, return_quantised=True)
    rng = np.random.default_rng(2)
    for b in rng.integers(0, B, 2):
        q_o, xs_o = O.quantize_rows_e4m3(X[b].float().numpy())
        assert np.array_equal(xs[b].cpu().numpy(), xs_o) and np.array_equal(Xq[b].cpu().view(torch.uint8).numpy(), q_o)
    Ybf = hk.expert_gather_fp8w_forward(Xg, Wqg, sg, Ig)
    for b, e in zip(rng.integers(0, B, 4), rng.integers(0, E, 4)):
        rows = X[b][Ind[b, e]].float().numpy()                               # [K, I]
        q_o, xs_o = O.quantize_rows_e4m3(rows)
        Xd = O.fp8_e4m3fn_to_float(q_o) * xs_o[:, None].astype(np.float64)
        W = O.dequant_fp8_weights(Wq[e:e + 1].view(torch.uint8).numpy(), scale[e:e + 1].numpy())[0]
        assert_close(Y[b, e], Xd @ W, torch.bfloat16, f"C5 fp8-act Y[{b},{e}]")
        ref = np64(Ybf[b, e])
        rel_rms = np.sqrt(((np64(Y[b, e]) - ref) ** 2).mean() / (ref ** 2).mean())
        assert rel_rms <= 5e-2, rel_rms
    assert torch.equal(Y, hk.expert_gather_fp8_forward(Xg, Wqg, sg, Ig))


def test_c2_inference_block_full_size():
    # gather -> relu -> scatter of the default shape in one kernel against the oracle's chained forward (rows rounded to
    # bf16 where a stored Y would be), repeated bit for bit, tokens nobody picked exactly zero
    cfg, inp, g = gpu_inputs("C2")
    B, T, E, K, I, J = cfg.dims
    got = hk.expert_mlp_forward(g["X"], g["Wg"], g["Ws"], g["Ind"], "relu", force_block=True)
    ref = O.mlp_forward(np64(inp["X"]), np64(inp["Wg"]), np64(inp["Ws"]), inp["Ind"].numpy(), T, "relu",
                        round_y=O.round_to_bf16)
    assert_close(got, ref, torch.bfloat16, "C2 inference block")
    assert torch.equal(got, hk.expert_mlp_forward(g["X"], g["Wg"], g["Ws"], g["Ind"], "relu", force_block=True))
    picked = torch.zeros(B, T, dtype=torch.bool)
    picked.scatter_(1, inp["Ind"].reshape(B, -1).long(), True)
    assert float(got.cpu()[~picked].abs().max() if (~picked).any() else 0.0) == 0.0
