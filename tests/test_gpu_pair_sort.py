"""Routing of prompts: the chosen experts, the offsets and the pairs' places."""
import ctypes as C

import pytest
import torch

from _util import gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,k,local", [
    (1, 1, 1, None), (63, 2, 2, None), (64, 8, 1, None), (1025, 16, 2, (4, 9)),      # one pair, ragged runs, a rank's share
    (9000, 16, 1, None), (300, 17, 2, (0, 17)), (2000, 64, 2, (10, 40)),             # each number of logits in registers
])
def test_pairs_go_to_their_experts(T, E, k, local):
    from vllm_hymeta import _C
    lib, g = _C.load(), gen(3)
    logits = torch.randn(T, E, generator=g).to(torch.bfloat16)
    if T > 60:
        logits[7] = float("nan")                     # picks valid experts
        logits[:, 0] += 2.0                          # uneven experts
    lo, hi = local or (0, E)
    d = logits.cuda()
    out = {n: torch.full((s,), -7, dtype=t, device="cuda") for n, s, t in (
        ("ids", T * k, torch.int32), ("weights", T * k, torch.float32), ("counts", E + 1, torch.int32), ("cursors", E + 1, torch.int32),
        ("offsets", E + 1, torch.int32), ("sorted", T * k, torch.int32), ("pos", T * k, torch.int32))}
    r = _C.MoeRouteArgs()
    ptr = lambda t: C.c_void_p(t.data_ptr())      # noqa: E731
    r.router_logits, r.topk_ids, r.topk_weights, r.counts, r.cursors = ptr(d), ptr(out["ids"]), ptr(out["weights"]), ptr(out["counts"]), ptr(out["cursors"])
    r.expert_offsets, r.sorted_pair, r.pair_pos = ptr(out["offsets"]), ptr(out["sorted"]), ptr(out["pos"])
    r.num_tokens, r.num_experts, r.top_k, r.logits_dtype, r.logits_stride_t = T, E, k, _C.HYMETA_BF16, E
    r.local_expert_begin, r.local_expert_end = lo, hi
    for _ in range(2):                               # the scratch words are anything
        assert lib.hymeta_moe_route(C.byref(r), None) == 0
    torch.cuda.synchronize()
    ids, pos, slots = out["ids"].cpu().long(), out["pos"].cpu(), out["sorted"].cpu()
    p, chosen = torch.softmax(logits.float(), -1).topk(k)
    good = ~torch.isnan(logits.float()).any(1)
    assert int(ids.min()) >= 0 and int(ids.max()) < E
    picked = torch.gather(logits.float(), 1, ids.view(T, k))
    assert torch.equal(picked[good], torch.gather(logits.float(), 1, chosen)[good])      # the same values (ties may name another index)
    assert torch.allclose(out["weights"].cpu().view(T, k)[good], p[good], rtol=2e-6, atol=0)
    counts = torch.bincount(ids, minlength=E)
    offsets = torch.cat((torch.zeros(1, dtype=torch.long), counts.cumsum(0)))
    assert torch.equal(out["offsets"].cpu().long(), offsets)
    here = (ids >= lo) & (ids < hi)
    assert bool((pos[~here] == -1).all())
    taken = pos[here].long()
    assert taken.unique().numel() == taken.numel()
    assert bool((taken >= offsets[ids[here]]).all() and (taken < offsets[ids[here] + 1]).all())
    assert torch.equal(slots[taken].long(), here.nonzero().flatten())
