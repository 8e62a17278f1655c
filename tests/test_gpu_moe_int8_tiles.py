"""Grouped int8 GEMMs of experts with many rows (tiles of 256 x 256) against exact integer products."""
import pytest
import torch

from _util import assert_bf16_ulp, gen, randn_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,H,inter", [
    ((1, 255, 256, 257, 0, 511), 256, 384),      # rows at and around the tile's edges, an expert without rows; 2 and 3 steps
    ((300, 84), 128, 256),                       # one step
    ((129, 700, 3), 512, 640),                   # several column tiles, the step loop's both parities
])
def test_experts_of_many_rows(sizes, H, inter):
    """Top-1 routing to experts of the given numbers of rows, in scattered order.  The int32 sums are exact and the scales,
    the routing weight and the one rounding are applied as below, so a value may differ by the routing weight's last fp32
    bit only: at most one bf16 ulp, and rarely."""
    from oracle.moe import moe_route_ref
    from vllm_hymeta import hip_ops

    E, T = len(sizes), sum(sizes)
    g = gen(11)
    x = randn_bf16(g, T, H)
    which = torch.repeat_interleave(torch.arange(E), torch.tensor(sizes))[torch.randperm(T, generator=g)]
    logits = randn_bf16(g, T, E, scale=0.25)
    logits[torch.arange(T), which] = 4.0
    w13 = torch.randint(-127, 128, (E, 2 * inter, H), generator=g, dtype=torch.int8)
    w2 = torch.randint(-127, 128, (E, H, inter), generator=g, dtype=torch.int8)
    s13 = (torch.rand(E, 2 * inter, generator=g) + 0.5) * (H ** -0.5 / 64)
    s2 = (torch.rand(E, H, generator=g) + 0.5) * (inter ** -0.5 / 64)
    out = hip_ops.moe_forward(x.cuda(), logits.cuda(), w13.cuda(), w2.cuda(), top_k=1, renormalize=False, w13_scale=s13.cuda(), w2_scale=s2.cuda())
    ids, wts = moe_route_ref(logits, 1, False)
    assert torch.equal(ids[:, 0].long(), which)
    xq, xs = (t.cpu() for t in hip_ops.w8a8_quantize(x.cuda()))
    ref = torch.zeros(T, H, dtype=torch.bfloat16)
    for e in range(E):
        rows = (which == e).nonzero().flatten()
        if rows.numel() == 0:
            continue
        h = (((xq[rows].long() @ w13[e].long().t()).float() * xs[rows, None]) * s13[e][None, :]).to(torch.bfloat16)
        aq, a_s = (t.cpu() for t in hip_ops.w8a8_quantize(hip_ops.silu_and_mul(h.cuda())))
        ref[rows] = ((((aq.long() @ w2[e].long().t()).float() * a_s[:, None]) * s2[e][None, :]) * wts[rows, 0:1]).to(torch.bfloat16)
    torch.cuda.synchronize()
    assert_bf16_ulp(out.cpu(), ref, "int8 experts", ulps=1)
    assert float((out.cpu() != ref).float().mean()) < 0.01
