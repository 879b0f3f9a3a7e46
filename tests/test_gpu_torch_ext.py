"""The C++ route of the launchers and autograd Functions (csrc/egs_torch.cpp) against the Python route: same bits for what it
takes, and what it does not take goes to the Python route."""
import pytest
import torch

from tests._util import make_case

pytestmark = pytest.mark.gpu

import expertscattergather_amd as egs
from expertscattergather_amd import _abi
from expertscattergather_amd import hip_kernels as hk

DEV = "cuda"
SHAPES = [(4, 64, 8, 16, 128, 64),       # one-kernel scatter with a routing table
          (1, 1, 1, 1, 1, 1),
          (3, 37, 5, 11, 29, 13),        # product rows through the workspace, odd sizes
          (2, 300, 4, 200, 256, 192)]


def step(case, dtype, ind, grad_of, mode, bias=False):
    B, T, E, K, I, J = case["shape"]
    g, s = egs.ExpertGather(E, I, J, bias=bias).to(DEV, dtype), egs.ExpertScatter(E, J, I, bias=bias).to(DEV, dtype)
    with torch.no_grad():
        g.W.copy_(case["Wg"]); s.W.copy_(case["Ws"])
        if bias:
            g.bias.copy_(case["X"][0, 0, :1].expand(E, 1, J) + torch.arange(E)[:, None, None]); s.bias.copy_(case["dOut"][0, 0].expand(E, 1, I))
    g.scatter_mode = s.scatter_mode = mode
    x = case["X"].to(DEV).requires_grad_(True)
    out = s(g(x, ind), ind, T)
    out.backward(grad_of(out))
    torch.cuda.synchronize()
    return (out.detach(), x.grad, g.W.grad, s.W.grad) + ((g.bias.grad, s.bias.grad) if bias else ())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("grad", ["dense", "expanded", "sliced"])
def test_the_two_routes_agree(shape, dtype, grad, monkeypatch):
    B, T, E, K, I, J = shape
    case = dict(make_case(5 + sum(shape), *shape, dtype), shape=shape)
    wide = torch.randn(B, T, I + 24, device=DEV).to(dtype)
    grad_of = {"dense": lambda out: case["dOut"].to(DEV), "expanded": lambda out: torch.ones((), device=DEV, dtype=dtype).expand(out.shape),
               "sliced": lambda out: wide[..., 8:8 + I]}[grad]
    ind_dtype = torch.int16 if dtype is torch.float16 else torch.int64
    mode = "compact" if grad == "sliced" else None
    Ind = case["Ind"].to(ind_dtype)
    assert _abi.torch_ext() is not None
    fast = step(case, dtype, Ind.to(DEV), grad_of, mode)
    monkeypatch.setattr(_abi, "_pycall", None)
    assert _abi.torch_ext() is None
    slow = step(case, dtype, Ind.to(DEV), grad_of, mode)
    for name, a, b in zip(("out", "dX", "dWg", "dWs"), fast, slow):
        assert torch.equal(a, b), name


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("shape", SHAPES + [(40, 30, 3, 30, 70, 33)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("mode", ["deterministic", "atomic"])
def test_biases_and_their_gradients(shape, dtype, mode, monkeypatch):
    """Added by the launch itself or by one of its own (csrc/egs_bias.hip), against the composition from torch operations; picks
    outside [0, T) bring no bias in the scatter, and one in the gather."""
    B, T, E, K, I, J = shape
    case = dict(make_case(19 + sum(shape), *shape, dtype), shape=shape)
    Ind = case["Ind"].clone()
    if E * K > 1:
        Ind[0, 0, 0], Ind[-1, -1, -1] = T, -1
    grad_of = lambda out: case["dOut"].to(DEV)
    fast = step(case, dtype, Ind.to(DEV), grad_of, mode, True)
    monkeypatch.setattr(_abi, "_pycall", None)
    slow = step(case, dtype, Ind.to(DEV), grad_of, mode, True)
    tol = {torch.float32: 2e-5, torch.float16: 4e-3, torch.bfloat16: 3e-2}[dtype]
    for name, a, b in zip(("out", "dX", "dWg", "dWs", "db_gather", "db_scatter"), fast, slow):
        assert a.shape == b.shape and a.dtype == b.dtype
        assert (a.float() - b.float()).abs().max() <= tol * b.float().abs().max(), name


@pytest.mark.parametrize("E", [3072, 3073, 6400])
def test_scatter_bias_is_rounded_once_for_any_number_of_experts(E):
    """bias_scatter_kernel counts the picks of 3072 experts at a time; what it adds to an output is still one fp32 sum."""
    B, T, K, I, J = 1, 3, 2, 40, 32
    gen = torch.Generator().manual_seed(E)
    Ind, bias = torch.randint(0, T, (B, E, K), generator=gen), (torch.rand(E, 1, I, generator=gen) + 0.5).bfloat16()
    Y, W = torch.zeros(B, E, K, J, dtype=torch.bfloat16), torch.zeros(E, J, I, dtype=torch.bfloat16)
    with _abi.launch_log() as log:
        out = hk.expert_scatter(Y.to(DEV), W.to(DEV), Ind.to(DEV), T, "deterministic", bias.to(DEV)).cpu().double()
    assert "bias_scatter_kernel" in log.kernels, log.kernels
    want = torch.zeros(T, I, dtype=torch.float64).index_add_(0, Ind.reshape(-1), bias[:, 0].double().repeat_interleave(K, 0))
    half_ulp = torch.exp2(torch.floor(torch.log2(want)) - 8)                     # 8 bits of significand
    assert ((out[0] - want).abs() <= half_ulp + E * K * 2.0 ** -24 * want).all()  # and an fp32 sum of E * K positive terms


def _fresh_table_case():
    shape = B, T, E, K, I, J = 8, 64, 16, 16, 128, 64       # (the smallest E whose gather backward reads the table)
    case = make_case(21, *shape, torch.bfloat16)
    x, W = case["X"].to(DEV).requires_grad_(True), case["Wg"].to(DEV).requires_grad_(True)
    Ind, other = case["Ind"].to(DEV), make_case(22, *shape, torch.bfloat16)["Ind"].to(DEV)
    dY = case["Y"].to(DEV)
    return x, W, Ind, other, dY, torch.autograd.grad(hk.expert_gather(x, W, other.clone()), (x, W), dY)


@pytest.mark.parametrize("remedy", ["invalidate", "switch off", "none"])
def test_gather_backward_uses_no_table_that_was_taken_back(remedy):
    """A write that the version counter does not see, between forward and backward, with either documented remedy: both gradients
    follow the indices as they are now.  (Without one the scatter in the backward still reads the table: it is in use.)"""
    x, W, Ind, other, dY, want = _fresh_table_case()
    y = hk.expert_gather(x, W, Ind)
    if remedy == "none":
        want = torch.autograd.grad(y, x, dY, retain_graph=True) + want[1:]
    assert hk._TABLE_ATTR in Ind.__dict__
    Ind.data.copy_(other)
    try:
        if remedy == "invalidate":
            hk.invalidate_routing_table(Ind)
        elif remedy == "switch off":
            hk.set_routing_table_cache(False)
        got = torch.autograd.grad(y, (x, W), dY)
    finally:
        hk.set_routing_table_cache(True)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_a_table_made_in_inference_mode():
    """It has no version to count up: no node holds it, taking it back works, and the gradients are the same."""
    x, W, Ind, other, dY, want = _fresh_table_case()
    with torch.inference_mode():
        hk.expert_gather(x, W, other)
    assert other.__dict__[hk._TABLE_ATTR][1].is_inference()
    y = hk.expert_gather(x, W, other)
    for a, b in zip(torch.autograd.grad(y, (x, W), dY, retain_graph=True), want):
        assert torch.equal(a, b)
    hk.invalidate_routing_table(other)
    for a, b in zip(torch.autograd.grad(y, (x, W), dY), want):
        assert torch.equal(a, b)


def test_captured_gather_backward_does_not_use_an_eager_table():
    """Forward eager, backward alone captured, indices rewritten between replays: every replay sorts what they then hold."""
    x, W, Ind, other, dY, want = _fresh_table_case()
    first = Ind.clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        torch.autograd.grad(hk.expert_gather(x, W, Ind.clone()), (x, W), dY)                # (library loading before the capture)
        y = hk.expert_gather(x, W, Ind)
        before = torch.autograd.grad(y, (x, W), dY, retain_graph=True)
    s.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        got = torch.autograd.grad(y, (x, W), dY, retain_graph=True)
    for ind, ref in ((first, before), (other, want), (first, before), (other, want)):
        Ind.data.copy_(ind)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(got, ref):
            assert torch.equal(a, b)
        (x.detach() * 2).sum().item()                                                       # other work between the replays


UNPACK = {"same": lambda t: t, "fp32": lambda t: t.float() if t.is_floating_point() else t.int(),
          "layout": lambda t: t.transpose(0, 1).contiguous().transpose(0, 1), "copy": lambda t: t.clone(),
          "alignment": lambda t: torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape).copy_(t)}


@pytest.mark.parametrize("bias", [False, True], ids=["plain", "bias"])
@pytest.mark.parametrize("unpack", list(UNPACK))
def test_saved_tensors_that_come_back_changed(unpack, bias, monkeypatch):
    """Saved-tensor hooks may hand back another type, layout or alignment: what the native nodes do not take goes the Python way."""
    shape = B, T, E, K, I, J = 4, 64, 8, 16, 128, 64
    case = dict(make_case(31, *shape, torch.bfloat16), shape=shape)
    case["Ind"][0, 0, 0], case["Ind"][-1, -1, -1] = T, -1

    def run():
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, UNPACK[unpack]):
            return step(case, torch.bfloat16, case["Ind"].to(DEV), lambda out: case["dOut"].to(DEV), None, bias)
    fast = run()
    monkeypatch.setattr(_abi, "_pycall", None)
    for name, a, b in zip(("out", "dX", "dWg", "dWs", "db_gather", "db_scatter"), fast, run()):
        assert a.dtype == b.dtype and a.shape == b.shape, name
        if bias:        # added in fp32 within a launch, or by torch to the rounded result
            assert (a.float() - b.float()).abs().max() <= 3e-2 * b.float().abs().max(), name
        else:
            assert torch.equal(a, b), name


def test_saved_tensors_that_come_back_on_the_cpu_are_refused_on_both_routes(monkeypatch):
    case = dict(make_case(32, 2, 20, 3, 4, 32, 32, torch.bfloat16), shape=(2, 20, 3, 4, 32, 32))
    for _ in range(2):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t.cpu()), pytest.raises(RuntimeError, match="no CPU fallback"):
            step(case, torch.bfloat16, case["Ind"].to(DEV), lambda out: case["dOut"].to(DEV), None)
        monkeypatch.setattr(_abi, "_pycall", None)


def test_autograd_contract_of_the_native_nodes():
    shape = B, T, E, K, I, J = 4, 64, 8, 16, 128, 64
    case = make_case(9, *shape, torch.bfloat16)
    x, W, Ind = case["X"].to(DEV).requires_grad_(True), case["Wg"].to(DEV), case["Ind"].to(DEV)
    y = hk.expert_gather(x, W, Ind)
    assert "Native" in y.grad_fn.name() and not hk.expert_gather(x.detach(), W, Ind).requires_grad
    with torch.no_grad():
        assert not hk.expert_gather(x, W, Ind).requires_grad
    y.sum().backward()                                  # W needs no gradient: only x gets one
    assert x.grad is not None and W.grad is None
    with pytest.raises(RuntimeError, match="second time"):
        y.sum().backward()
    y = hk.expert_gather(x, W, Ind)
    Ind[0, 0, 0] = (Ind[0, 0, 0] + 1) % T               # a saved tensor written in place is noticed
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t, lambda t: t):
        y = hk.expert_gather(x, W, Ind)
    assert len(packed) >= 3
    y.sum().backward()


def test_what_the_native_route_declines_goes_the_python_way():
    shape = B, T, E, K, I, J = 2, 40, 4, 8, 64, 32
    case = make_case(11, *shape, torch.float32)
    X, W, Ind = case["X"].to(DEV), case["Wg"].to(DEV), case["Ind"].to(DEV)
    ext = _abi.torch_ext()
    call = lambda x, w, i, t=torch.float32: ext.gather_forward(x, w, i, t, 0, False, False, None)
    assert call(X, W, Ind) is not None
    off = torch.empty(X.numel() + 1, device=DEV)[1:].view_as(X).copy_(X)
    for args in [(X.transpose(0, 1).contiguous().transpose(0, 1), W, Ind), (off, W, Ind), (X.bfloat16(), W, Ind), (X.cpu(), W, Ind),
                 (X, W, Ind.float()), (X, W, Ind, torch.bfloat16), (X[:0], W, Ind[:0]), (X, W[:3], Ind)]:
        assert call(*args) is None
    assert torch.equal(hk.expert_gather(off, W, Ind), hk.expert_gather(X, W, Ind))
    with pytest.raises(ValueError):
        hk.expert_gather(X, W[:3], Ind)
    with torch.autograd.forward_ad.dual_level(), pytest.raises(Exception):      # no forward-mode derivative, on either route
        hk.expert_gather(torch.autograd.forward_ad.make_dual(X, torch.ones_like(X)), W, Ind)
