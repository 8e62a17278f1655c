"""The delta rule's slices of value columns, by every way to cut them, and portions too short for a chunk beside longer ones:
against the recurrence in 64 bits."""
import pytest
import torch

from _util import gen

pytestmark = pytest.mark.gpu
EDGES = [8, 63, 64, 65, 7, 129, 2, 1, 130, 3, 127, 128]


def _recurrence(q, k, v, beta, l2, state, starts, context, slots, scale, eps):
    group = v.shape[1] // q.shape[1]
    q, k = (x.double().repeat_interleave(group, 1) for x in (q, k))
    q = q / torch.sqrt(q.square().sum(-1, keepdim=True) + eps) * scale
    k = k / torch.sqrt(k.square().sum(-1, keepdim=True) + eps)
    beta, decay, v, out, states = torch.sigmoid(beta.double()), torch.exp2(l2.double()), v.double(), [], state.double().clone()
    for s in range(len(starts) - 1):
        S = states[slots[s]].clone() if slots[s] >= 0 and context[s] > 0 else torch.zeros_like(states[0])
        for t in range(starts[s], starts[s + 1]):
            S = S * decay[t][:, None, None]
            u = beta[t][:, None] * (v[t] - torch.einsum("hdv,hd->hv", S, k[t]))
            S = S + k[t][:, :, None] * u[:, None]
            out.append(torch.einsum("hdv,hd->hv", S, q[t]))
        if slots[s] >= 0:
            states[slots[s]] = S
    return torch.stack(out), states


@pytest.mark.parametrize("D,Dv,H,Hk,lens,shift", [
    (32, 96, 4, 2, EDGES, 0),                    # slices of 32, shorter portions in a launch of their own
    (128, 64, 4, 4, EDGES + [1] * 60, 1),        # the same, values at odd addresses
    (96, 192, 4, 2, EDGES, 0),                   # slices of 64
    (128, 128, 4, 1, [300, 7, 1] + [70] * 12, 0),
    (64, 128, 24, 8, EDGES, 0), (128, 256, 16, 8, EDGES, 0),          # slices of 128
    (64, 128, 2, 1, [200], 0), (128, 32, 2, 2, [65, 5], 0),           # slices of 16
    (96, 96, 16, 4, EDGES, 0), (96, 128, 24, 8, EDGES, 0), (32, 128, 24, 8, EDGES, 0),        # slices of 32, and of 128 with other heads
    (96, 96, 4, 2, [300, 65], 0), (32, 32, 4, 4, [200, 9, 1], 0),      # slices of 16 whose blocks do not deal evenly over the waves
    (128, 128, 4, 2, [2, 7, 1, 3, 6], 0), (256, 64, 2, 2, [2, 5], 0),  # nothing long enough for a chunk
    (32, 64, 4, 4, [5, 1, 7], 1), (64, 32, 2, 1, [3, 7], 0), (96, 64, 2, 2, [1, 6, 2], 0), (96, 32, 2, 2, [2, 4], 0),
    # short portions in a launch of their own beside chunks: by their number, as the others fill the chip, by their rows
    (96, 64, 32, 8, [70, 8] + [1, 3, 7] * 46, 0), (128, 128, 32, 8, [40] + [1] * 36, 0), (64, 64, 16, 16, [40] + [7] * 25, 0),
    (32, 64, 32, 8, [70, 8] + [1, 3, 7] * 46, 0),        # ... and as many that stay
])
def test_every_slice_against_64_bits(D, Dv, H, Hk, lens, shift):
    """Operands from fp32 enter as two bf16 parts, 2^-17 of the operand each, a few such roundings on the way to an output and
    their growth over three chunks: 2e-5 of the norm."""
    from vllm_hymeta import hip_ops
    T, n, g = sum(lens), len(lens), gen(D + Dv + len(lens))
    q, k = (torch.randn(T, Hk, D, generator=g).bfloat16() for _ in range(2))
    v = torch.randn(T * H * Dv + shift, generator=g).bfloat16()
    beta, l2 = torch.randn(T, H, generator=g).bfloat16(), -torch.rand(T, H, generator=g) * 0.2
    state = torch.randn(n, H, D, Dv, generator=g) * 0.1
    starts, context, slots = [sum(lens[:i]) for i in range(n + 1)], [5 * (i % 2) for i in range(n)], [i if i != 3 else -1 for i in range(n)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    dev, got = "cuda", state.cuda()
    out = hip_ops.delta_rule(q.to(dev), k.to(dev), v.to(dev)[shift:].view(T, H, Dv), beta.to(dev), l2.to(dev), got, i32(starts), i32(context), i32(slots), max(lens), D ** -0.5, 1e-6)
    want, states = _recurrence(q, k, v[shift:].view(T, H, Dv), beta, l2, state, starts, context, slots, D ** -0.5, 1e-6)
    out, got = out.view(T, H, Dv).double().cpu(), got.double().cpu()
    for s in range(n):
        a, b = starts[s], starts[s + 1]
        assert float((out[a:b] - want[a:b]).norm() / want[a:b].norm()) < 2e-5, s
    assert float((got - states).norm() / states.norm()) < 2e-5
    assert torch.equal(got[3:4], state[3:4].double()) if n > 3 else True


def test_a_portion_longer_than_the_bound_says():
    """A bound of fewer rows than a chunk takes asks for no workspace: every row goes token by token, however many there are."""
    from vllm_hymeta import hip_ops
    H, D, lens, g = 4, 128, [3, 70, 1, 130], gen(7)
    T, n, starts = sum(lens), len(lens), [sum(lens[:i]) for i in range(len(lens) + 1)]
    q, k, v = (torch.randn(T, H, D, generator=g).bfloat16() for _ in range(3))
    beta, l2, state = torch.randn(T, H, generator=g).bfloat16(), -torch.rand(T, H, generator=g) * 0.2, torch.randn(n, H, D, D, generator=g) * 0.1
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    got = state.cuda()
    out = hip_ops.delta_rule(q.cuda(), k.cuda(), v.cuda(), beta.cuda(), l2.cuda(), got, i32(starts), i32([1] * n), i32(list(range(n))), 4, D ** -0.5, 1e-6)
    want, states = _recurrence(q, k, v, beta, l2, state, starts, [1] * n, list(range(n)), D ** -0.5, 1e-6)
    assert float((out.view(T, H, D).double().cpu() - want).norm() / want.norm()) < 2e-6        # (fp32 throughout)
    assert float((got.double().cpu() - states).norm() / states.norm()) < 2e-6
