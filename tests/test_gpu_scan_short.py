"""Portions too short for a chunk of the lightning attention and the decay scan, beside longer ones and alone: against the
recurrence in 64 bits."""
import pytest
import torch

from _util import gen

pytestmark = pytest.mark.gpu
MIXED = [7, 1, 8, 2, 65, 3, 1, 130, 6]


def _recurrence(q, k, v, w, decay, state, starts, context, slots):
    out, states = [], state.double().clone()
    for s in range(len(starts) - 1):
        S = states[slots[s]].clone() if slots[s] >= 0 and context[s] > 0 else torch.zeros_like(states[0])
        for t in range(starts[s], starts[s + 1]):
            S = S * decay[t][:, None, None] + k[t][:, :, None] * w[t][:, None]
            out.append((S * q[t][:, :, None]).sum(1))
        if slots[s] >= 0:
            states[slots[s]] = S
    return torch.stack(out), states


@pytest.mark.parametrize("silu", [True, False])
@pytest.mark.parametrize("D,Dv,H,lens", [
    (128, 128, 14, MIXED + [100] * 6), (64, 64, 4, MIXED), (32, 96, 4, MIXED), (128, 256, 4, [2, 7, 1, 3]),
    (64, 128, 2, [700, 1, 5, 300]),               # cut into segments
    (64, 128, 32, [40] * 4 + [1] * 26 + [7, 2, 3, 6, 5]),         # in a launch beside the chunks'
])
def test_short_portions(D, Dv, H, lens, silu):
    """Rows of portions of up to 7 stay in fp32: 1e-6 of the norm.  The others' operands enter as two bf16 parts, 2e-5, behind a
    silu rounded to bf16 on the way, 3e-3."""
    from vllm_hymeta import hip_ops
    T, n, g = sum(lens), len(lens), gen(D + Dv + silu)
    Hk = H if silu else H // 2
    qkv = torch.randn(T, 2 * Hk * D + H * Dv, generator=g).bfloat16()
    q, k, v = (x.unflatten(1, (h, d)) for x, h, d in zip(qkv.split([Hk * D, Hk * D, H * Dv], 1), (Hk, Hk, H), (D, D, Dv)))
    state, decay = torch.randn(n, H, D, Dv, generator=g) * 0.1, 1 - torch.rand(H, generator=g) * 0.1
    l2, b, skip = -torch.rand(T, H, generator=g) * 0.2, torch.rand(T, H, generator=g), torch.randn(H, generator=g)
    starts, context, slots = [sum(lens[:i]) for i in range(n + 1)], [5 * (i % 2) for i in range(n)], [i if i != 3 else -1 for i in range(n)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    got, dev, where = state.cuda(), qkv.cuda(), (i32(starts), i32(context), i32(slots), max(lens))
    if silu:
        out = hip_ops.lightning_attention(dev, got, decay.cuda(), H, D, Dv, *where)
        act = torch.nn.functional.silu
        want, states = _recurrence(act(q.double()), act(k.double()), act(v.double()), act(v.double()), decay.double().expand(T, H), state, starts, context, slots)
    else:
        dq, dk, dv = (x.unflatten(1, (h, d)) for x, h, d in zip(dev.split([Hk * D, Hk * D, H * Dv], 1), (Hk, Hk, H), (D, D, Dv)))
        out = hip_ops.decay_scan(dq, dk, dv, got, *where, log2_decay=l2.cuda(), v_scale=b.cuda(), skip=skip.cuda())
        qd, kd, vd = q.double().repeat_interleave(2, 1), k.double().repeat_interleave(2, 1), v.double()
        want, states = _recurrence(qd, kd, vd, vd * b.double()[:, :, None], torch.exp2(l2.double()), state, starts, context, slots)
        want = want + skip.double()[None, :, None] * vd
    out, got = out.view(T, H, Dv).double().cpu(), got.double().cpu()
    for s in range(n):
        rows, bound = slice(starts[s], starts[s + 1]), 1e-6 if lens[s] < 8 else 3e-3 if silu else 2e-5
        assert float((out[rows] - want[rows]).norm() / want[rows].norm()) < bound, s
        assert slots[s] < 0 or float((got[s] - states[s]).norm() / states[s].norm()) < bound, s
    assert torch.equal(got[3], state[3].double())


@pytest.mark.parametrize("silu", [True, False])
def test_sequences_without_rows_have_no_slot(silu):
    """Their slots lie far outside the state, which is neither read nor written for them: outputs and states as without them."""
    from vllm_hymeta import hip_ops
    D, H, g = 64, 2, gen(9)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    qkv, state, decay = torch.randn(75, 3 * H * D, generator=g).bfloat16().cuda(), torch.randn(2, H, D, D, generator=g).cuda(), torch.tensor([0.9, 0.99]).cuda()
    q, k, v = (x.unflatten(1, (H, D)) for x in qkv.split([H * D] * 3, 1))
    results = []
    for starts, slots in (([0, 5, 75], [0, 1]), ([0, 0, 5, 5, 75, 75], [1 << 30, 0, 1 << 30, 1, 1 << 30])):
        got, where = state.clone(), (i32(starts), i32([3] * len(slots)), i32(slots), 70)
        out = hip_ops.lightning_attention(qkv, got, decay, H, D, D, *where) if silu else hip_ops.decay_scan(q, k, v, got, *where, decay=decay)
        results.append((out, got))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])


@pytest.mark.parametrize("silu", [True, False])
@pytest.mark.parametrize("D,Dv,H", [(128, 128, 28), (64, 128, 64)])
def test_single_rows_whose_states_do_not_fit_the_cache(D, Dv, H, silu):
    """256 sequences, one of them of two rows: a launch of its own, fewer workgroups of which share a compute unit.  In 64 bits on
    the GPU."""
    from vllm_hymeta import hip_ops
    n, g = 256, torch.Generator(device="cuda").manual_seed(D + H)
    new = lambda *shape: torch.empty(*shape, device="cuda").normal_(generator=g)  # noqa: E731
    qkv, state, decay = new(n + 1, H * (2 * D + Dv)).bfloat16(), new(n, H, D, Dv) * 0.1, 1 - 0.1 * new(H).abs().clamp_max(1)
    q, k, v = (x.unflatten(1, (H, d)) for x, d in zip(qkv.split([H * D, H * D, H * Dv], 1), (D, D, Dv)))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    where, S = (i32([0, 2] + list(range(3, n + 2))), i32([4] * n), i32(list(range(n))), 2), state.double()
    out = (hip_ops.lightning_attention(qkv, state, decay, H, D, Dv, *where) if silu else hip_ops.decay_scan(q, k, v, state, *where, decay=decay)).view(n + 1, H, Dv)
    q, k, v = (torch.nn.functional.silu(x.double()) if silu else x.double() for x in (q, k, v))
    d = decay.double()[:, None, None]
    first = S[0] * d + k[0][:, :, None] * v[0][:, None]
    assert float((out[0] - torch.matmul(q[0][:, None], first)[:, 0]).norm() / out[0].norm()) < 1e-6
    S[0] = first
    S = S * d + k[1:][..., None] * v[1:][:, :, None]
    want = torch.matmul(q[1:][:, :, None], S)[:, :, 0]
    assert float((out[1:] - want).norm() / want.norm()) < 1e-6 and float((state - S).norm() / S.norm()) < 1e-6
