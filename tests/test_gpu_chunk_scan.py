"""Chunks of 64 rows of linear attention with decays at the edges of its kernel: numbers of rows around the chunk's and the
segments', every width of a workgroup, against the recurrence in 64 bits token by token."""
import pytest
import torch

from _util import gen

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _recurrence(q, k, v, log2_decay, b, skip, state, lens, carried):
    """``q, k [T, H, D]``, ``v [T, H, Dv]``, ``log2_decay, b [T, H]``, all fp64 -> outputs and the states after."""
    out, after, t = [], [], 0
    for s, rows in enumerate(lens):
        S = state[s].clone() if carried[s] else torch.zeros_like(state[s])
        for _ in range(rows):
            S = S * torch.exp2(log2_decay[t])[:, None, None] + k[t][:, :, None] * (b[t][:, None] * v[t])[:, None, :]
            out.append((q[t][:, :, None] * S).sum(1) + skip[:, None] * v[t])
            t += 1
        after.append(S)
    return torch.stack(out), torch.stack(after)


def _layout(lens, carried):
    starts = torch.tensor([0] + lens).cumsum(0).int()
    return [x.to(DEV) for x in (starts, torch.tensor([7 if c else 0 for c in carried], dtype=torch.int32), torch.arange(len(lens), dtype=torch.int32))]


def _rel(x, ref):
    return float((x.double().cpu().reshape(ref.shape) - ref).norm() / ref.norm())


# widths: 8, 4 and 2 waves to a workgroup, one and two slices; portions below a chunk, at its edges, in segments (576 rows and
# more of few heads) with a short last segment, and beside portions that are shorter than a segment or than a chunk
SHAPES = [
    (128, 128, 2, [8, 63, 64, 65]), (128, 128, 32, [130, 9, 64, 100]), (128, 256, 2, [577, 40]), (64, 64, 3, [576, 640, 8]),
    (32, 32, 2, [1, 200, 600, 7]), (64, 96, 2, [129, 701]), (32, 128, 24, [70, 64, 9, 65, 66]), (128, 64, 2, [1200]),
    # a long portion among single rows and short ones; long ones side by side, whose cuts have neighbouring numbers
    (128, 128, 2, [1] * 9 + [1300] + [1] * 20 + [600, 7, 8, 400]), (32, 32, 2, [705, 1, 700, 1, 577, 640, 1]),
    # eight multiplying and eight staging waves over segments: with the states chained by the segments themselves, in two slices of the
    # columns, and by a launch of their own (eleven segments)
    (128, 128, 20, [1300, 7, 300, 1]), (64, 128, 24, [5, 1217, 600]), (128, 256, 10, [1300, 600]), (128, 128, 12, [2112]),
    (64, 128, 40, [9, 64, 65, 128, 127, 8, 3]),
    # the shortest segments: of one chunk, with the least rows that are cut and one fewer; beside as many single rows as leave 192 rows each
    (128, 128, 28, [192, 1, 65]), (128, 128, 28, [191]), (64, 128, 16, [520, 40]), (128, 64, 8, [193, 192, 191, 64]), (32, 32, 64, [577] + [1] * 64),
    (32, 32, 64, [577, 300] + [1] * 64),
]


@pytest.mark.parametrize("D,Dv,H,lens", SHAPES)
def test_plain_and_per_row_decays(D, Dv, H, lens):
    """bf16 inputs enter the products exactly and everything in fp32 as two bf16 parts (an error of 2^-17 of the operand at
    most); the sum over a portion's terms keeps that relative size: 2e-5 of the result's norm allows for the decays' rounding."""
    from vllm_hymeta import hip_ops
    T, S, Hk = sum(lens), len(lens), 1 if H % 2 else H // 2
    g = gen(D + Dv + H)
    q, k, v = (torch.randn(T, n, d, generator=g).bfloat16() for n, d in ((Hk, D), (Hk, D), (H, Dv)))
    state, carried = torch.randn(S, H, D, Dv, generator=g), [i % 2 == 0 for i in range(S)]
    l2, b, skip = -torch.rand(T, H, generator=g) * 0.2, torch.rand(T, H, generator=g) + 0.5, torch.randn(H, generator=g)
    decay = torch.rand(H, generator=g) * 0.2 + 0.8
    starts, context, slots = _layout(lens, carried)
    rep = lambda x: x.double().repeat_interleave(H // Hk, 1)
    for per_row in (True, False):
        got = state.to(DEV)
        kw = dict(log2_decay=l2.to(DEV), v_scale=b.to(DEV), skip=skip.to(DEV)) if per_row else dict(decay=decay.to(DEV))
        out = hip_ops.decay_scan(q.to(DEV), k.to(DEV), v.to(DEV), got, starts, context, slots, max(lens), **kw)
        one = torch.ones(T, H, dtype=torch.float64)
        ref, after = _recurrence(rep(q), rep(k), v.double(), l2.double() if per_row else one * torch.log2(decay.double()), b.double() if per_row else one,
                                 skip.double() if per_row else torch.zeros(H, dtype=torch.float64), state.double(), lens, carried)
        assert _rel(out, ref) < 2e-5 and _rel(got, after) < 2e-5, (per_row, _rel(out, ref), _rel(got, after))


@pytest.mark.parametrize("D,Dv,H,lens", SHAPES)
def test_lightning(D, Dv, H, lens):
    """Queries, keys and values through their silu, rounded to bf16 where they are a product's operands: 2^-9 each, so
    2 x 2^-9 of the result's norm bounds the independent errors of the factors of one term (portions under 8 rows and steps
    keep fp32)."""
    from vllm_hymeta import hip_ops
    T, S = sum(lens), len(lens)
    g = gen(D + Dv + H + 1)
    qkv = torch.randn(T, H * (2 * D + Dv), generator=g).bfloat16()
    state, carried = torch.randn(S, H, D, Dv, generator=g), [i % 2 == 0 for i in range(S)]
    decay = torch.rand(H, generator=g) * 0.2 + 0.8
    starts, context, slots = _layout(lens, carried)
    got = state.to(DEV)
    out = hip_ops.lightning_attention(qkv.to(DEV), got, decay.to(DEV), H, D, Dv, starts, context, slots, max(lens))
    x = torch.nn.functional.silu(qkv.double())
    one = torch.ones(T, H, dtype=torch.float64)
    ref, after = _recurrence(x[:, :H * D].reshape(T, H, D), x[:, H * D:2 * H * D].reshape(T, H, D), x[:, 2 * H * D:].reshape(T, H, Dv),
                             one * torch.log2(decay.double()), one, torch.zeros(H, dtype=torch.float64), state.double(), lens, carried)
    assert _rel(out, ref) < 2 ** -8 and _rel(got, after) < 2 ** -8, (_rel(out, ref), _rel(got, after))


@pytest.mark.parametrize("D,Dv,H,lens", [(128, 128, 2, [64, 200]), (64, 96, 2, [1300]), (32, 64, 3, [65, 8])])
def test_lightning_state_holds_keys_in_two_parts(D, Dv, H, lens):
    """The states against silu(k) in 64 bits and silu(v) as the bf16 it is rounded to: the keys' two parts leave 2^-17 of an
    operand.  The silu's own error, 2^-21, flips the rounding of about 2^-12 of the values by 2^-8 of the value: 2^-14 of the
    norm.  Twice their sum; keys in one part would leave 2^-9 / sqrt(3)."""
    from vllm_hymeta import hip_ops
    T, S = sum(lens), len(lens)
    g = gen(D + Dv + H + 2)
    qkv = torch.randn(T, H * (2 * D + Dv), generator=g).bfloat16()
    state, carried = torch.randn(S, H, D, Dv, generator=g), [i % 2 == 0 for i in range(S)]
    decay = torch.rand(H, generator=g) * 0.2 + 0.8
    starts, context, slots = _layout(lens, carried)
    got = state.to(DEV)
    hip_ops.lightning_attention(qkv.to(DEV), got, decay.to(DEV), H, D, Dv, starts, context, slots, max(lens))
    x = torch.nn.functional.silu(qkv.double())
    one = torch.ones(T, H, dtype=torch.float64)
    _, after = _recurrence(x[:, :H * D].reshape(T, H, D), x[:, H * D:2 * H * D].reshape(T, H, D), x[:, 2 * H * D:].bfloat16().double().reshape(T, H, Dv),
                           one * torch.log2(decay.double()), one, torch.zeros(H, dtype=torch.float64), state.double(), lens, carried)
    assert _rel(got, after) < 2 * (2 ** -17 + 2 ** -14), _rel(got, after)
