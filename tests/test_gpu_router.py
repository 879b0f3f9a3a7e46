"""The one-kernel expert-choice router (csrc/egs_router.hip) against torch on the CPU: the same tokens in the same order, at sizes
where a wavefront's column, the row loads or the selection have remainders; ties, and what stays with torch."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from expertscattergather_amd import _abi
from expertscattergather_amd.router import expert_choice_router

SHAPES = [(1, 1, 1, 1), (3, 17, 5, 4), (2, 64, 9, 64), (2, 65, 64, 33), (64, 256, 32, 32), (1, 1024, 60, 100), (2, 1025, 3, 257), (1, 4096, 20, 512),
          (1, 257, 7, 129), (64, 300, 33, 20), (1, 4097, 17, 65), (40, 1025, 17, 65)]
LARGE = [(1, 1024, 70, 100), (1, 700, 140, 30), (2, 3000, 40, 130), (64, 800, 129, 9)]


def kernels_of(B, T, E):
    """What a call launches: the rows' sums ahead of the router where it asks for a workspace to put them."""
    return ["router_stats_kernel", "router_kernel"] if _abi.lib().egs_expert_choice_router_workspace_bytes(B, T, E) > 0 else ["router_kernel"]


def without_workspace(logits, K, ind_dtype):
    """The router as one launch: every workgroup computes the rows' sums."""
    B, T, E = logits.shape
    Ind, scores = torch.empty(B, E, K, dtype=ind_dtype, device="cuda"), torch.empty(B, E, K, device="cuda")
    codes = {torch.float32: _abi.F32, torch.float16: _abi.F16, torch.bfloat16: _abi.BF16}, {torch.int16: _abi.IND_I16, torch.int64: _abi.IND_I64}
    with _abi.launch_log() as log:
        rc = _abi.lib().egs_expert_choice_router(logits.data_ptr(), Ind.data_ptr(), scores.data_ptr(), None, 0, B, T, E, K, codes[0][logits.dtype],
                                                 codes[1][ind_dtype], torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and log.kernels == ["router_kernel"], (rc, log.kernels)
    return Ind, scores


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("B,T,E,K", SHAPES, ids=lambda v: str(v))
def test_router_matches_topk(B, T, E, K, dtype):
    gen = torch.Generator().manual_seed(B + T + E + K)
    logits = torch.randn(B, T, E, generator=gen).to(dtype)
    ind_dtype = torch.int16 if dtype is torch.float16 else torch.int64
    on_device = logits.cuda()
    with _abi.launch_log() as log:
        Ind, scores = expert_choice_router(on_device, K, ind_dtype)
    assert log.kernels == kernels_of(B, T, E) and Ind.dtype is ind_dtype and scores.dtype is torch.float32
    if len(log.kernels) > 1:                            # one launch, whatever the library prefers: the same bits
        assert all(torch.equal(a, b) for a, b in zip((Ind, scores), without_workspace(on_device, K, ind_dtype)))
    aff = torch.softmax(logits.double(), -1).transpose(1, 2)
    want = aff.topk(K, -1)[0]
    Ind, scores = Ind.cpu().long(), scores.cpu()
    assert ((Ind >= 0) & (Ind < T)).all() and (Ind.sort(-1)[0].diff(dim=-1) > 0).all()
    assert torch.allclose(scores.double(), want, rtol=1e-5, atol=0)
    assert torch.allclose(scores.double(), aff.gather(-1, Ind), rtol=1e-5, atol=0)
    assert (scores.diff(dim=-1) <= 0).all()


@pytest.mark.parametrize("B,T,E,K", LARGE, ids=lambda v: str(v))
def test_large_logits_have_their_row_sums_first(B, T, E, K):
    logits = torch.randn(B, T, E, generator=torch.Generator().manual_seed(T))
    logits[0, 3, 1] = float("nan")
    with _abi.launch_log() as log:
        Ind, scores = expert_choice_router(logits.cuda(), K)
    assert log.kernels == ["router_stats_kernel", "router_kernel"]
    assert (Ind[0, :, 0] == 3).all() and scores[0, :, 0].isnan().all()
    aff = torch.softmax(logits.double(), -1).transpose(1, 2).nan_to_num(9.0)
    scores = scores.cpu().double().nan_to_num(9.0)
    assert torch.allclose(scores, aff.topk(K, -1)[0], rtol=1e-5, atol=0) and torch.allclose(scores, aff.gather(-1, Ind.cpu()), rtol=1e-5, atol=0)


def test_ties_take_the_lowest_tokens_and_a_nan_comes_first():
    logits = torch.zeros(2, 100, 3)
    logits[1, 40] = float("nan")
    Ind, scores = expert_choice_router(logits.cuda(), 7)
    assert Ind[0].tolist() == [[0, 1, 2, 3, 4, 5, 6]] * 3
    assert Ind[1].tolist() == [[40, 0, 1, 2, 3, 4, 5]] * 3 and torch.isnan(scores[1, :, 0]).all()


def test_gradients_and_strided_logits_stay_with_torch():
    logits = torch.randn(2, 33, 4, device="cuda", requires_grad=True)
    with _abi.launch_log() as log:
        Ind, scores = expert_choice_router(logits, 5)
        expert_choice_router(logits.detach().transpose(0, 1), 2)
    assert log.kernels == []
    scores.sum().backward()
    assert logits.grad is not None
    fast, _ = expert_choice_router(logits.detach(), 5)
    assert torch.equal(fast, Ind)


@pytest.mark.parametrize("B,T,E,K", [(2, 129, 64, 7), (9, 300, 33, 20), (3, 513, 5, 60), (2, 769, 9, 5), (3, 1025, 41, 12), (2, 2049, 8, 39), (1, 3073, 10, 70),
                                     (1, 4097, 3, 9), (1, 8193, 5, 300)], ids=lambda v: str(v))
def test_row_sums_first_or_by_every_workgroup(B, T, E, K):
    """Sizes that need no workspace and are faster with one, and columns of one chunk more than each length that wavefronts hold: the same bits."""
    logits = torch.randn(B, T, E, generator=torch.Generator().manual_seed(T)).to(torch.bfloat16).cuda()     # with ties
    logits[0, 3, 1] = float("nan")
    L, stream = _abi.lib(), torch.cuda.current_stream().cuda_stream
    need = L.egs_expert_choice_router_workspace_bytes(B, T, E)
    assert need in (0, B * T * 8)
    with _abi.launch_log() as log:
        Ind, scores = expert_choice_router(logits, K)
    assert log.kernels == kernels_of(B, T, E), log.kernels
    own_Ind, own = without_workspace(logits, K, torch.int64)
    if need == 0:                                       # a workspace that is not asked for changes nothing
        ws, more_Ind, more = torch.empty(B * T * 8, dtype=torch.uint8, device="cuda"), torch.empty_like(Ind), torch.empty_like(scores)
        with _abi.launch_log() as log:
            assert L.egs_expert_choice_router(logits.data_ptr(), more_Ind.data_ptr(), more.data_ptr(), ws.data_ptr(), ws.numel(), B, T, E, K, _abi.BF16,
                                              _abi.IND_I64, stream) == 0
        assert log.kernels == ["router_kernel"] and torch.equal(more_Ind, own_Ind)
    assert torch.equal(Ind, own_Ind) and torch.equal(scores.view(torch.int32), own.view(torch.int32))
    aff = torch.softmax(logits.cpu().double(), -1).transpose(1, 2).nan_to_num(9.0)
    scores = scores.cpu().double().nan_to_num(9.0)
    assert torch.allclose(scores, aff.topk(K, -1)[0], rtol=1e-5, atol=0) and torch.allclose(scores, aff.gather(-1, Ind.cpu()), rtol=1e-5, atol=0)
