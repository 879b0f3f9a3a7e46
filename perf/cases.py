"""Measured cases of the expert gather / scatter path: what programs built on this package ask of it, through its modules,
its router, its inference block and its fp8 gathers.

A case is one pass of such a program: a training step through the modules and autograd, a forward pass without gradients,
a routed expert layer, or the forward of a layer whose gather weights are stored in fp8.  Sizes are those of the
benchmark configurations, of the sweeps and of the tests (which draw every dimension at random, odd ones included)."""
import math

import torch

import expertscattergather_amd as egs
from expertscattergather_amd import hip_kernels, workloads
from expertscattergather_amd.router import expert_choice_router

DEVICE = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
IND_DTYPES = {"int16": torch.int16, "int32": torch.int32, "int64": torch.int64}


def _case(kind, B, T, E, K, I, J, dtype, **options):
    return dict({"kind": kind, "B": B, "T": T, "E": E, "K": K, "I": I, "J": J, "dtype": dtype}, **options)


def _train(*args, routing="uniform", ind="int64", mode="deterministic", bias=False):
    return _case("train", *args, routing=routing, ind=ind, mode=mode, bias=bias)


def _infer(*args, routing="uniform", ind="int64", mode="deterministic"):
    return _case("infer", *args, routing=routing, ind=ind, mode=mode)


def _layer(*args, activation="relu", train=False):
    return _case("layer", *args, activation=activation, train=train)


def _fp8(*args, activations="bf16"):
    return _case("fp8", *args, activations=activations)


def listed():
    cases = {
        # a small model or a debugging run: four sequences of 64 tokens; launches and host work are all there is
        "smoke_train_bf16": _train(4, 64, 8, 16, 128, 64, "bf16"),
        # the default shape, a training step in bf16 with indices as a router gives them: the headline configuration
        "default_train_bf16": _train(64, 256, 32, 32, 128, 64, "bf16"),
        # the default shape as the sweeps time it: fp32, int16 indices drawn with replacement
        "default_train_f32": _train(64, 256, 32, 32, 128, 64, "f32", routing="replacement", ind="int16"),
        # the default shape in fp32, forward only
        "default_infer_f32": _infer(64, 256, 32, 32, 128, 64, "f32"),
        # an expert-choice layer at the default shape when the model is served: router, then the block
        "routed_layer_bf16": _layer(64, 256, 32, 32, 128, 64, "bf16"),
        # sizes nobody rounded, as the tests draw them from 1..127; fp32, with biases
        "ragged_train_f32": _train(53, 97, 29, 41, 111, 75, "f32", routing="replacement", ind="int32", bias=True),
        # the widest point of the sweep over I
        "wide_train_bf16": _train(64, 256, 32, 32, 768, 64, "bf16", routing="replacement", ind="int16"),
        # a mid-sized fp16 model whose sizes fill no tile
        "uneven_train_f16": _train(6, 1100, 20, 150, 328, 136, "f16"),
        # Zipf-distributed routing: hot tokens repeat within and across experts
        "zipf_train_bf16": _train(16, 1024, 64, 128, 512, 128, "bf16", routing="zipf"),
        # long sequences, fine-grained experts
        "long_train_bf16": _train(8, 4096, 128, 256, 1024, 256, "bf16"),
        # large fp8 weights, few rows for each expert (generation): the weights' bytes count
        "fp8_decode": _fp8(4, 512, 256, 8, 2048, 512, "bf16"),
        # the same layer over whole prompts: the largest call
        "fp8_prefill": _fp8(32, 2048, 256, 64, 2048, 512, "bf16"),
    }
    return [dict(case, name=name) for name, case in cases.items()]


MOST_FLOPS = 2 * 8 * 128 * 256 * 1024 * 256           # of one product of a drawn step: the long-sequence configuration's
MOST_FP8_FLOPS = 2 * 32 * 256 * 64 * 2048 * 512       # of one product of a drawn fp8 pass: the largest configuration's


def _log_int(rng, low, high):
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _width(rng, low, high):
    """A feature dimension: usually a multiple of 32, as in models, sometimes any number, as in the tests."""
    n = _log_int(rng, low, high)
    return n if rng.random() < 0.4 else max(32, round(n / 32) * 32)


def draw(rng):
    kind = rng.choices(["train", "infer", "layer", "fp8"], [11, 3, 3, 3])[0]
    while True:
        if kind == "fp8":
            B, T, E = _log_int(rng, 1, 32), _log_int(rng, 64, 2048), _log_int(rng, 16, 256)
            K = _log_int(rng, 4, min(64, T))
            I, J = 128 * _log_int(rng, 2, 16), 16 * _log_int(rng, 4, 32)
            most = MOST_FP8_FLOPS
        else:
            B, T, E = _log_int(rng, 1, 128), _log_int(rng, 32, 4096), _log_int(rng, 4, 128)
            K = _log_int(rng, 4, min(256, T))
            I, J = _width(rng, 24, 1024), _width(rng, 16, 256)
            most = MOST_FLOPS
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        work = workloads.flops((B, T, E, K, I, J)) * (8 if dtype == "f32" and kind != "fp8" else 1)    # fp32 products run at a lower rate
        if work <= most and B * T * I <= 8 * 4096 * 1024 * (4 if kind == "fp8" else 1):
            break
    dims = (B, T, E, K, I, J)
    routing = rng.choice(["uniform", "uniform", "replacement", "zipf"])
    ind = rng.choice(["int64", "int64", "int32", "int16"])
    mode = rng.choices(["deterministic", "atomic", "compact"], [8, 1, 1])[0]
    if kind == "train":
        return _train(*dims, dtype, routing=routing, ind=ind, mode=mode, bias=rng.random() < 0.15)
    if kind == "infer":
        return _infer(*dims, dtype, routing=routing, ind=ind, mode=mode)
    if kind == "layer":
        return _layer(*dims, dtype, activation=rng.choice(["relu", "gelu", "silu"]), train=rng.random() < 0.3)
    return _fp8(*dims, "bf16", activations=rng.choice(["bf16", "fp8"]))


def _dims(case):
    return tuple(case[k] for k in ("B", "T", "E", "K", "I", "J"))


def _routing(case, gen):
    """Ind [B,E,K]: distinct tokens per expert as from a router, drawn with replacement, or Zipf-distributed."""
    B, T, E, K, _, _ = _dims(case)
    kind = case.get("routing", "uniform")
    if kind == "uniform":
        ind = torch.stack([torch.rand(E, T, device=DEVICE, generator=gen).argsort(dim=-1)[:, :K] for _ in range(B)])
    elif kind == "replacement":
        ind = torch.randint(0, T, (B, E, K), device=DEVICE, generator=gen)
    else:
        cdf = torch.arange(1, T + 1, device=DEVICE, dtype=torch.float64).pow(-1.2).cumsum(0)
        ranks = torch.searchsorted(cdf / cdf[-1], torch.rand(B, E, K, device=DEVICE, dtype=torch.float64, generator=gen))
        ind = torch.randperm(T, device=DEVICE, generator=gen)[ranks.clamp_max(T - 1)]
    return ind.to(IND_DTYPES[case.get("ind", "int64")]).contiguous()


def prepare(case, seed):
    B, T, E, K, I, J = _dims(case)
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    dt = DTYPES[case["dtype"]]

    def normal(*shape, scale=1.0, dtype=dt):
        return torch.randn(*shape, device=DEVICE, generator=gen).mul_(scale).to(dtype)

    state = {"case": dict(case), "x": normal(B, T, I)}
    if case["kind"] == "layer":
        state["logits"] = normal(B, T, E, dtype=torch.float32)
    else:
        state["Ind"] = _routing(case, gen)
    w_gather, w_scatter = normal(E, I, J, scale=I ** -0.5), normal(E, J, I, scale=J ** -0.5)
    if case["kind"] == "fp8":
        state["w_gather"], state["scale"] = workloads.quantize_fp8_weights(w_gather)
        state["w_scatter"] = w_scatter
        return state
    if case["kind"] == "layer":
        state["w_gather"], state["w_scatter"] = w_gather, w_scatter
        if case["train"]:
            state["d_out"] = normal(B, T, I)
            for k in ("x", "w_gather", "w_scatter"):
                state[k].requires_grad_(True)
        return state
    bias = case.get("bias", False)
    with torch.device(DEVICE):
        gather, scatter = egs.ExpertGather(E, I, J, bias=bias).to(dt), egs.ExpertScatter(E, J, I, bias=bias).to(dt)
    with torch.no_grad():
        gather.W.copy_(w_gather)
        scatter.W.copy_(w_scatter)
        if bias:
            gather.bias.copy_(normal(E, 1, J, scale=0.1))
            scatter.bias.copy_(normal(E, 1, I, scale=0.1))
    gather.scatter_mode = scatter.scatter_mode = case["mode"]
    state["gather"], state["scatter"] = gather, scatter
    if case["kind"] == "train":
        state["x"].requires_grad_(True)
        state["d_out"] = normal(B, T, I)
    return state


def run(state):
    case = state["case"]
    T = case["T"]
    if case["kind"] == "layer":
        Ind, scores = expert_choice_router(state["logits"], case["K"])
        x, w_gather, w_scatter = state["x"], state["w_gather"], state["w_scatter"]
        if not case["train"]:
            with torch.no_grad():
                return {"out": hip_kernels.expert_mlp_forward(x, w_gather, w_scatter, Ind, case["activation"]), "Ind": Ind, "scores": scores}
        x.grad = w_gather.grad = w_scatter.grad = None
        out = hip_kernels.expert_mlp(x, w_gather, w_scatter, Ind, case["activation"])
        out.backward(state["d_out"])
        return {"out": out.detach(), "Ind": Ind, "scores": scores, "x": x.grad, "w_gather": w_gather.grad, "w_scatter": w_scatter.grad}

    Ind = state["Ind"]
    # every batch of a real program brings indices of its own; the state's are used again, so what an earlier pass left with them goes
    hip_kernels.invalidate_routing_table(Ind)
    if case["kind"] == "fp8":
        gather = hip_kernels.expert_gather_fp8_forward if case["activations"] == "fp8" else hip_kernels.expert_gather_fp8w_forward
        Y = gather(state["x"], state["w_gather"], state["scale"], Ind)
        return {"Y": Y, "out": hip_kernels.expert_scatter_forward_call(Y, state["w_scatter"], Ind, T, torch.float32)}

    x, gather, scatter = state["x"], state["gather"], state["scatter"]
    if case["kind"] == "infer":
        with torch.no_grad():
            Y = gather(x, Ind)
            return {"Y": Y, "out": scatter(Y, Ind, T)}
    x.grad = None
    gather.zero_grad(set_to_none=True)
    scatter.zero_grad(set_to_none=True)
    out = scatter(gather(x, Ind), Ind, T)
    out.backward(state["d_out"])
    grads = {"x": x.grad}
    for name, module in (("gather", gather), ("scatter", scatter)):
        grads.update({name + "." + p: q.grad for p, q in module.named_parameters()})
    return dict(grads, out=out.detach())


def work(case):
    B, T, E, K, I, J = dims = _dims(case)
    size = 4 if case["dtype"] == "f32" else 2
    picks, tokens, weights = B * E * K, B * T, E * I * J
    rows_read = min(tokens, picks) * I * size
    indices = picks * (2 if case.get("ind") == "int16" else 4 if case.get("ind") == "int32" else 8)
    out = tokens * I * size
    biases = E * (I + J) * size if case.get("bias") else 0
    if case["kind"] == "fp8":
        return {"bytes": rows_read + weights * (1 + size) + E * J * 4 + indices + picks * J * size + out, "flops": 2 * workloads.flops(dims)}
    moved = rows_read + 2 * weights * size + biases + out
    if case["kind"] == "layer":
        moved += tokens * E * 4 + picks * (8 + 4)              # logits in; indices and scores out
    else:
        moved += indices
    if case["kind"] == "infer":
        moved += picks * J * size                              # Y is an output
    if case["kind"] == "train" or case.get("train"):
        moved += rows_read + out + 2 * weights * size + biases  # d_out in; the gradients out
        return {"bytes": moved, "flops": 6 * workloads.flops(dims)}
    return {"bytes": moved, "flops": 2 * workloads.flops(dims)}


def tolerance(case):
    rel = {"f32": 1e-5, "f16": 2e-3, "bf16": 1e-2}[case["dtype"]]
    if case["kind"] == "layer":
        # two affinities closer than fp32 resolves may change places in the router's order (and one of them its place in the top K)
        return {"rel": max(rel, 2e-3), "differ": 1e-3}
    return {"rel": rel}
