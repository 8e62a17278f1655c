"""Grouped products of 4-bit GPTQ experts of more than a few rows: the kernel of 64-slot tiles against 64-bit sums and, bit for bit,
against the kernel of 32-slot tiles (which a larger number of experts behind the pairs asks for)."""
import ctypes as C

import pytest
import torch

from _util import gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,K,N,group,f16,zero_offset,div,local", [
    # slots at the edges of the tiles, an expert without; one group, fewer groups than four classes, uneven classes; one step more
    # and fewer than are copied ahead
    ((1, 64, 65, 0, 128, 129, 200), 128, 128, 128, True, 1, 1, (0, 7)),
    ((1, 64, 65, 0, 128, 129, 200), 64, 256, 64, False, 1, 1, (0, 7)),
    ((1, 64, 65, 0, 128, 129, 200), 384, 384, 128, False, 0, 2, (0, 7)),
    ((33, 100, 31, 63), 320, 128, 64, True, 0, 3, (1, 4)),
    ((33, 100, 31, 63), 1152, 256, 128, True, 1, 1, (0, 3)),
    ((300,), 448, 640, 64, False, 1, 1, (0, 1)),
    ((40, 0, 60) * 24, 256, 128, 128, True, 1, 2, (2, 71)),      # more experts than lanes
])
def test_grouped_gptq_products(sizes, K, N, group, f16, zero_offset, div, local):
    from vllm_hymeta import _C
    lib, E, P = _C.load(), len(sizes), sum(sizes)
    g = gen(31)
    kind = torch.float16 if f16 else torch.bfloat16
    T = (P + div - 1) // div
    q, z = torch.randint(0, 16, (E, K, N), generator=g), torch.randint(0, 16, (E, K // group, N), generator=g)
    scale = ((torch.rand(E, K // group, N, generator=g) + 0.5) * 0.01).to(kind)
    packed = sum(q[:, i::8].long() << (4 * i) for i in range(8))
    zeros = sum(z[:, :, i::8].long() << (4 * i) for i in range(8))
    as_int = lambda t: torch.where(t >= 2 ** 31, t - 2 ** 32, t).int().contiguous().cuda()      # noqa: E731
    x = torch.randn(T, K, generator=g).bfloat16()
    slots, order = torch.randperm(T * div, generator=g)[:P].int(), torch.randperm(P, generator=g).int()
    factor = torch.rand(P, generator=g) + 0.5
    offsets = torch.tensor([0] + list(sizes)).cumsum(0).int()
    d = [t.cuda() for t in (x, scale, slots, order, factor, offsets)] + [as_int(packed), as_int(zeros)]
    outs = []
    for experts in (0, 1 << 20):
        out = torch.full((P + 1, N), 7.0, dtype=torch.bfloat16, device="cuda")
        a = _C.MoeGptqGemmArgs()
        a.x, a.scales, a.a_rows, a.scale_rows, a.row_scale, a.expert_offsets, a.qweight, a.qzeros = (t.data_ptr() for t in d)
        a.out, a.a_rows_div, a.max_rows, a.K, a.N, a.bits, a.group_size, a.zero_offset = out.data_ptr(), div, P, K, N, 4, group, zero_offset
        a.scales_dtype = _C.HYMETA_F16 if f16 else _C.HYMETA_BF16
        a.local_expert_begin, a.local_expert_end = local
        a.x_stride_m, a.out_stride_m = K, N
        assert lib.hymeta_moe_gptq_gemm_rank(C.byref(a), experts, torch.cuda.current_stream().cuda_stream) == 0
        outs.append(out)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
    w = scale.double().repeat_interleave(group, 1) * (q - (z + zero_offset).repeat_interleave(group, 1)).double()
    out = outs[0].cpu()
    for e in range(E):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        if not local[0] <= e < local[1]:
            assert bool((out[lo:hi] == 7.0).all())
            continue
        rows = x[(slots[lo:hi] // div).long()].double()
        f = factor[order[lo:hi].long()].double()[:, None]
        ref = rows @ w[e] * f
        # fp32 sums of x (128 + q) and of x times 128 + z, at most 160 |x| a term each, of which rounding leaves 2^-24; then one to bf16
        bound = 2.0 ** -8 * ref.abs() + 2.0 ** -24 * 160 * 2 * (rows.abs() @ scale[e].double().repeat_interleave(group, 0)) * f
        assert bool(((out[lo:hi].double() - ref).abs() <= bound).all()), f"expert {e}"
    assert bool((out[P] == 7.0).all())
