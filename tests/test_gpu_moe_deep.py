"""Grouped products of experts that do not fill a tile of 256 slots, bit for bit on small integers (test_gpu_tile_gemm.py's
problem): every sum is exact and one rounding to bf16 remains."""
import ctypes as C

import pytest
import torch

from _util import gen

from test_gpu_tile_gemm import CLAMPED, NONE, SILU, SILU_EXACT, _activate, _ints

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,K,N,div,local,act,int8", [
    # slots at the edges of 64, 128 and 192, an expert without; fewer steps than are copied ahead, and just as many
    ((1, 64, 65, 128, 129, 0, 192, 193, 63), 64, 5120, 1, (0, 9), NONE, False),
    ((1, 64, 65, 128, 129, 0, 192, 193, 63), 192, 5120, 2, (0, 9), SILU, False),
    ((1, 64, 65, 128, 129, 0, 192, 193, 63), 320, 5248, 1, (0, 9), CLAMPED, False),
    ((1, 64, 65, 128, 129, 0, 192, 193, 63), 384, 5120, 1, (2, 8), SILU_EXACT, False),
    ((1, 64, 65, 128, 129, 0, 192, 193, 63), 128, 5120, 2, (0, 9), NONE, True),
    ((1, 64, 65, 128, 129, 0, 192, 193, 63), 896, 5120, 1, (2, 8), SILU, True),
    ((256, 257, 1, 2, 3, 513, 40, 8), 576, 5248, 1, (0, 8), NONE, False),       # tiles of 256, two and three an expert
    ((256, 257, 1, 2, 3, 513, 40, 8), 256, 5248, 3, (0, 8), SILU, True),
    ((130, 257, 127), 448, 128, 1, (0, 3), NONE, False),                        # one column: tiles of 64 slots
    ((130, 257, 0, 255), 256, 2048, 2, (0, 4), SILU, True),                     # tiles of 128
    ((300, 640), 192, 384, 1, (0, 2), SILU, False),                             # many slots of few columns
    ((9, 0, 17, 64, 70) * 15, 128, 256, 1, (0, 75), NONE, False),               # more experts than lanes
    ((9, 0, 17, 64, 70) * 15, 256, 128, 1, (3, 74), SILU, True),
])
def test_experts_below_a_tile(sizes, K, N, div, local, act, int8):
    from vllm_hymeta import _C
    lib, E, P = _C.load(), len(sizes), sum(sizes)
    g = gen(9)
    kind, T, cols = torch.int8 if int8 else torch.bfloat16, (sum(sizes) + div - 1) // div, N // 2 if act else N
    x, w = _ints(g, -3, 3, T, K).to(kind).cuda(), _ints(g, -2, 2, E, N, K).to(kind).cuda()
    slots, order = torch.randperm(T * div, generator=g)[:P].int().cuda(), torch.randperm(P, generator=g).int().cuda()
    factor, x_scale, w_scale = (2.0 ** _ints(g, -2, 1, *shape).float().cuda() for shape in ((P,), (T,), (E, N)))
    offsets = torch.tensor([0] + list(sizes)).cumsum(0)
    on_card, out = offsets.int().cuda(), torch.full((P + 1, cols), 7.0, dtype=torch.bfloat16, device="cuda")
    a = _C.MoeGemmArgs()
    a.x, a.weights, a.out, a.expert_offsets = x.data_ptr(), w.data_ptr(), out.data_ptr(), on_card.data_ptr()
    a.a_rows, a.a_rows_div, a.scale_rows, a.row_scale = slots.data_ptr(), div, order.data_ptr(), factor.data_ptr()
    a.max_rows, a.K, a.N, a.x_stride_m, a.out_stride_m, a.w_stride_e = P, K, N, K, cols, N * K
    a.local_expert_begin, a.local_expert_end = local
    if int8:
        a.operand_dtype, a.x_scale, a.w_scale = _C.HYMETA_I8, x_scale.data_ptr(), w_scale.data_ptr()
    assert lib.hymeta_moe_gemm_glu_takes(C.byref(a), E) == 1
    assert lib.hymeta_moe_gemm_glu(C.byref(a), E, act, 7.0, 1.702, torch.cuda.current_stream().cuda_stream) == 0
    source = (slots // div).long()
    for e in range(E):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        s = source[lo:hi]
        h = x[s].float() @ w[e].float().t()                          # exact: |sums| < 2^24
        if int8:
            h = h * x_scale[s][:, None] * w_scale[e]
        h = (h * factor[order[lo:hi].long()][:, None]).to(torch.bfloat16)
        assert torch.equal(out[lo:hi], _activate(h, act) if hi > lo and local[0] <= e < local[1] else torch.full_like(out[lo:hi], 7.0)), f"expert {e}"
    assert bool((out[P] == 7.0).all())
