"""The routers' scores and choice with their sums formed by halves that trade places: tokens, outputs and columns that do not fill their
rounds, against 64-bit sums."""
import ctypes as C

import pytest
import torch

from _util import gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,K,top", [(1, 1, 3, 1), (3, 8, 256, 2), (5, 9, 257, 3), (4, 17, 1030, 17), (2, 1024, 64, 4), (9, 63, 3584, 2)])
def test_scores_and_choice(T, E, K, top):
    from vllm_hymeta import _C
    lib, g = _C.load(), gen(T + E + K)
    x, w = torch.randn(T, K, generator=g).bfloat16(), torch.randn(E, K, generator=g) * K ** -0.5
    xd, wd = x.cuda(), w.cuda()
    ids, weights = torch.zeros(T, top, dtype=torch.int32, device="cuda"), torch.zeros(T, top, device="cuda")
    offsets, pairs, pos = (torch.zeros(n, dtype=torch.int32, device="cuda") for n in (E + 1, T * top, T * top))
    a = _C.MoeRouteSigmoidArgs()
    a.x, a.router_weight, a.topk_ids, a.topk_weights, a.expert_offsets, a.sorted_pair, a.pair_pos = (
        t.data_ptr() for t in (xd, wd, ids, weights, offsets, pairs, pos))
    a.num_tokens, a.num_experts, a.top_k, a.hidden, a.act_dtype, a.scale, a.x_stride_t = T, E, top, K, _C.HYMETA_BF16, 1.0, K
    assert lib.hymeta_moe_route_sigmoid(C.byref(a), torch.cuda.current_stream().cuda_stream) == 0
    score = torch.sigmoid(x.double() @ w.double().t())
    picked = ids.cpu().long()
    assert all(len(set(row)) == top for row in picked.tolist())
    best = score.topk(top).values
    # a fp32 sum of K terms in 256 strands: 2^-24 (K / 256 + 8) of the terms' absolute sum, a quarter of it in the score
    slack = 2.0 ** -24 * (K / 256 + 10) * (x.double().abs() @ w.double().abs().t()).max().item() + 2.0 ** -22
    assert float((score.gather(1, picked) - best).abs().max()) <= slack
    assert float((weights.cpu().double() - best / (best.sum(1, keepdim=True) + 1e-20)).abs().max()) <= 4 * slack
    assert int(offsets[-1]) == T * top


@pytest.mark.parametrize("T,E,K,top", [(1, 1, 8, 1), (3, 15, 2056, 2), (2, 17, 4104, 2), (5, 33, 256, 1), (256, 64, 520, 2)])
def test_one_launch_router(T, E, K, top):
    """Logits against 64 bits; choice, weights and the sort against the kernel's own bf16 logits.  The last token's row is NaN."""
    from vllm_hymeta import _C
    lib, g = _C.load(), gen(T * E + K)
    x, w = torch.randn(T, K, generator=g).bfloat16(), (torch.randn(E, K, generator=g) * K ** -0.5).bfloat16()
    x[-1, 0] = float("nan")
    xd, wd = x.cuda(), w.cuda()
    ids, weights, logits = torch.full((T, top), -9, dtype=torch.int32, device="cuda"), torch.zeros(T, top, device="cuda"), torch.zeros(T, E, dtype=torch.bfloat16, device="cuda")
    offsets, pairs, pos, ticket = (torch.zeros(n, dtype=torch.int32, device="cuda") for n in (E + 1, T * top, T * top, 16))
    a = _C.MoeRouterArgs()
    a.x, a.gate_weight, a.logits_out, a.topk_ids, a.topk_weights, a.expert_offsets, a.sorted_pair, a.pair_pos, a.ticket = (
        t.data_ptr() for t in (xd, wd, logits, ids, weights, offsets, pairs, pos, ticket))
    a.x_stride_t, a.num_tokens, a.num_experts, a.top_k, a.renormalize, a.hidden = K, T, E, top, 0, K
    a.local_expert_begin, a.local_expert_end = 0, E
    for _ in range(2):                                       # the ticket is ready again
        assert lib.hymeta_moe_router(C.byref(a), torch.cuda.current_stream().cuda_stream) == 0
    own, live = logits.cpu(), T - 1
    exact = x[:live].double() @ w.double().t()
    # fp32 sums of K terms in 256 strands, then one rounding to bf16
    slack = 2.0 ** -8 * exact.abs() + 2.0 ** -24 * (K / 256 + 10) * (x[:live].double().abs() @ w.double().abs().t())
    assert bool(((own[:live].double() - exact).abs() <= slack).all())
    left, soft = own[:live].double().clone(), torch.softmax(own[:live].double(), 1)
    picked = ids.cpu().long()
    for k in range(top):
        first = torch.tensor([int((row == row.max()).nonzero()[0]) for row in left], dtype=torch.long)
        assert torch.equal(picked[:live, k], first)
        assert torch.allclose(weights.cpu().double()[:live, k], soft.gather(1, first[:, None])[:, 0], rtol=2e-6, atol=0)
        left.scatter_(1, first[:, None], -float("inf"))
    assert picked[-1].tolist() == list(range(top)) and bool(torch.isnan(weights[-1]).all())
    counts = torch.bincount(picked.flatten(), minlength=E)
    assert torch.equal(offsets.cpu().long(), torch.cat([torch.zeros(1, dtype=torch.long), counts.cumsum(0)]))
    order = pairs.cpu().long()
    assert torch.equal(order.sort().values, torch.arange(T * top)) and torch.equal(picked.flatten()[order], picked.flatten().sort().values)
    assert torch.equal(order[pos.cpu().long()], torch.arange(T * top))


@pytest.mark.parametrize("E,top,mode", [(3, 3, "sigmoid"), (70, 9, "sigmoid"), (5, 2, "softmax"), (130, 66, "softmax")])
def test_scores_that_are_no_numbers(E, top, mode):
    """A token whose scores are all NaN, or -inf but for one: experts that exist, each once, with weights that say so."""
    from vllm_hymeta import _C
    lib, g, T, K = _C.load(), gen(E), 6, 64
    x, w, bias = torch.randn(T, K, generator=g).bfloat16(), torch.randn(E, K, generator=g) * K ** -0.5, torch.zeros(E)
    x[2, 5] = x[5, 0] = float("nan")
    if mode == "softmax":
        bias[:] = -float("inf")
        bias[E - 2] = 0.0
    xd, wd, bd = x.cuda(), w.cuda(), bias.cuda()
    ids, weights = torch.full((T, top), -9, dtype=torch.int32, device="cuda"), torch.zeros(T, top, device="cuda")
    offsets, pairs, pos = (torch.full((n,), -9, dtype=torch.int32, device="cuda") for n in (E + 1, T * top, T * top))
    a = _C.MoeRouteSigmoidArgs()
    a.x, a.router_weight, a.router_bias, a.topk_ids, a.topk_weights, a.expert_offsets, a.sorted_pair, a.pair_pos = (
        t.data_ptr() for t in (xd, wd, bd, ids, weights, offsets, pairs, pos))
    a.num_tokens, a.num_experts, a.top_k, a.hidden, a.act_dtype, a.scale, a.x_stride_t = T, E, top, K, _C.HYMETA_BF16, 1.0, K
    a.score_mode = _C.ROUTE_SOFTMAX_CHOSEN if mode == "softmax" else _C.ROUTE_SIGMOID_SUM
    assert lib.hymeta_moe_route_sigmoid(C.byref(a), torch.cuda.current_stream().cuda_stream) == 0
    picked, weights = ids.cpu(), weights.cpu()
    assert bool(((picked >= 0) & (picked < E)).all()) and all(len(set(row)) == top for row in picked.tolist())
    assert torch.equal(torch.isnan(weights), torch.isnan(x).any(1)[:, None].expand(T, top))
    live = [t for t in range(T) if t not in (2, 5)]
    if mode == "softmax":
        assert bool((picked[live, 0] == E - 2).all()) and torch.equal(weights[live], torch.eye(1, top).expand(len(live), top))
    else:
        best = torch.sigmoid(x[live].double() @ w.double().t()).topk(top).values
        assert torch.allclose(weights[live].double(), best / best.sum(1, keepdim=True), rtol=0, atol=1e-5)
    assert int(offsets[-1]) == T * top and sorted(pos.cpu().tolist()) == list(range(T * top))
