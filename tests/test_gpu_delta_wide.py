"""The delta rule over many (portion, head) pairs runs in slices of 128 value columns: against the same sequences one at a
time, which run in narrow slices.  A long portion among single rows runs in narrow slices too."""
import pytest
import torch

from _util import gen

pytestmark = pytest.mark.gpu
DEV = "cuda"


EDGES = [8, 63, 64, 65, 130, 7, 128, 129, 20, 1, 130, 97, 126, 127, 128]        # worth ten portions of 130: 160 wide slices


@pytest.mark.parametrize("D,Dv,H,Hk,lens", [
    (32, 128, 16, 4, EDGES), (64, 256, 8, 8, EDGES), (96, 128, 16, 16, EDGES), (128, 128, 16, 8, EDGES),
    (128, 128, 16, 8, [1] * 20 + [300] + [1] * 12 + [9, 130]), (96, 128, 12, 12, [1] * 20 + [300] + [1] * 12 + [9, 130]),
    (128, 128, 16, 8, [1] * 60 + [300] + [1] * 30),
    # more pairs than half of the compute units: the shortest sequences whole, the others' halves side by side; 80, 136 and 104 whole
    (128, 128, 28, 14, [300, 257, 299, 260, 321, 270]), (128, 128, 28, 14, [300, 290, 257, 260, 299, 270, 5]), (64, 256, 15, 15, [257] * 6),
    (32, 128, 28, 28, [300] * 5), (96, 128, 28, 28, [300] * 6 + [7]),      # and a portion too short for a chunk where none is expected:
    (128, 128, 28, 14, [300] * 6 + [7]), (64, 128, 28, 7, [64] * 8 + [3]), (128, 128, 16, 16, [64, 64, 64, 5]), (128, 96, 12, 4, [64, 64, 64, 5]),
    # a chunk's sequence found in two round trips and in three
    (64, 64, 4, 4, [1] * 40 + [70] + [1] * 24 + [64, 130] + [1] * 63 + [9]), (32, 32, 2, 2, [1] * 66 + [65] + [1] * 4100 + [130, 3])])
def test_wide_slices_equal_narrow_ones(D, Dv, H, Hk, lens):
    """Both multiply the same operands (fp32 as two bf16 parts, 2^-17 of the operand) and add in another order: 1e-5 of the
    norm covers what that rounding grows to over a few chunks.  Rows at a chunk's edges, several chunks, a portion that goes
    token by token, carried states and one sequence without a slot."""
    from vllm_hymeta import hip_ops
    T, S = sum(lens), len(lens)
    g = gen(D + Dv)
    q, k, v = (torch.randn(T, n, d, generator=g).bfloat16().to(DEV) for n, d in ((Hk, D), (Hk, D), (H, Dv)))
    beta = torch.randn(T, H, generator=g).bfloat16().to(DEV)
    l2 = (-torch.rand(T, H, generator=g) * 0.2).to(DEV)
    state = (torch.randn(S, H, D, Dv, generator=g) * 0.1).to(DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    context, slots = [5 if i % 2 else 0 for i in range(S)], [i if i != 3 else -1 for i in range(S)]
    wide, narrow = state.clone(), state.clone()
    starts = [sum(lens[:i]) for i in range(S + 1)]
    out = hip_ops.delta_rule(q, k, v, beta, l2, wide, i32(starts), i32(context), i32(slots), max(lens), D ** -0.5, 1e-6)
    for s in range(S):
        a, b = starts[s], starts[s + 1]
        one = hip_ops.delta_rule(q[a:b], k[a:b], v[a:b], beta[a:b], l2[a:b], narrow, i32([0, b - a]), i32(context[s:s + 1]), i32(slots[s:s + 1]), b - a, D ** -0.5, 1e-6)
        assert float((out[a:b] - one).norm() / one.norm()) < 1e-5, s
        assert float((wide[s] - narrow[s]).norm() / narrow[s].norm()) < 1e-5, s
