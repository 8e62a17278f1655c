"""The router's scores and choice with its sums formed by halves that trade places: tokens, outputs and columns that do not fill its
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
