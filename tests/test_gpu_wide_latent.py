"""Attention over latent rows of 256 / 384 / 512 + 64 (one pass over the keys for all value columns) at the edges of its tiles:
128 (query, head) rows a workgroup, 32 keys a tile in a prompt, 64 in four runs of 16 in a decode step, 16 query heads a slice;
pages that hold a tile and pages that do not.

Bound: the outputs are bf16 (2^-9 of each value at most); the weights are two bf16 parts (2^-17), exponentials and products
fp32 (below 2^-12 over these lengths); together below 2^-9 + 2^-11 in the norm."""
from itertools import accumulate

import pytest
import torch

pytestmark = pytest.mark.gpu
BOUND = 2.0 ** -9 + 2.0 ** -11


def reference(q, rows, C, scale, sink, window, keep, chunk, softcap, bias, gate, ctx):
    """One sequence in 64 bits: q [n, H, C + 64] at positions ctx .. over rows [ctx + n, C + 64]."""
    n, H, _ = q.shape
    i, j = torch.arange(ctx, ctx + n)[:, None], torch.arange(ctx + n)
    seen = j <= i
    if chunk:
        seen = seen & (j >= i // chunk * chunk)
    elif window:
        seen = seen & ((j > i - window) | (j < keep))
    s = torch.einsum("nhd,jd->hnj", q, rows) * scale
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    if bias is not None:
        s = s - bias[:, None, None] * torch.log1p(0.25 * (i - j).clamp_min(0).double())
    s = s.masked_fill(~seen, float("-inf"))
    if sink is not None:
        s = torch.cat((s, sink[:, None, None].expand(H, n, 1)), -1)
    p = torch.softmax(s, -1)[..., :ctx + n].nan_to_num()      # (no keys: 0)
    o = torch.einsum("hnj,jc->nhc", p, rows[:, :C])
    return o if gate is None else o * torch.sigmoid(gate)[:, :, None]


@pytest.mark.parametrize("C,H,page,lens,ctxs,opts", [
    (512, 16, 64, [8, 1, 9], [0, 4096, 120], {}),                            # a whole block of rows, one row more, decode
    (512, 28, 64, [33, 1, 1], [31, 63, 64], dict(sink=True)),                # two head slices, the last of 12
    (512, 17, 8, [5, 1], [3, 15], dict(sink=True)),                          # pages smaller than a tile, a slice of one head
    (384, 3, 32, [150, 1, 2], [0, 200, 1], dict(window=70, keep=5)),         # kept first keys ahead of the window
    (256, 4, 16, [64, 1, 1], [65, 0, 129], dict(chunk=48, gate=True)),
    (512, 1, 128, [129, 1], [0, 511], dict(softcap=5.0, bias=True)),
    (512, 16, 64, [3, 1, 1], [100, 127, 0], dict(sink=True, gate=True)),      # few keys: single rows among the portions' blocks
    (384, 5, 16, [2, 1, 1], [100, 128, -1], {}),                              # one key past that
    (512, 16, 64, [1, 3, 20, 1], [-1, -1, -10, 300], {}),                    # rows in front of their sequence
    (256, 4, 16, [1, 70, 2], [-1, -30, -2], dict(chunk=20, sink=True)),
    # keys cut into slices beside single rows: a window, kept first keys, a gate; some blocks whole
    (512, 16, 64, [9, 1, 3, 1], [2500, 700, 5, 64], dict(window=1600, keep=40, gate=True, sink=True)),
    (256, 40, 16, [1, 5, 1], [900, 1400, 31], dict(chunk=700, gate=True)),
    (256, 33, 64, [1] * 5, [0, 15, 16, 1000, 63], dict(sink=True, window=33)),
    *[(c, 16, 64, [1, 1], [64 * n - 1, 20], dict(sink=True, gate=True)) for c, n in ((384, 2), (512, 3), (256, 8), (512, 9))],      # partials of a row
    # as many of 128 columns as a thread takes at once, four or eight, and one more; statistics for two each
    *[(c, 16, 64, [1], [64 * n - 1], dict(sink=True, gate=True)) for c, n in ((512, 16), (384, 17), (256, 32), (512, 33), (512, 129))],
    # as many (row, head) pairs as are merged in parts of the columns, and a row more
    (512, 16, 64, [29, 1], [2000, 300], dict(sink=True)), (384, 16, 64, [30, 1], [2000, 300], dict(sink=True, gate=True)), (512, 16, 64, [30, 1], [2000, 5], {}),
])
def test_against_64_bits(C, H, page, lens, ctxs, opts):
    from vllm_hymeta import hip_ops
    g = torch.Generator().manual_seed(C + H)
    D = C + 64
    o = dict(dict(sink=False, window=0, keep=0, chunk=0, softcap=0.0, bias=False, gate=False), **opts)
    rows = [torch.randn(n + c, D, generator=g).bfloat16() for n, c in zip(lens, ctxs)]
    q = [torch.randn(n, H, D, generator=g).bfloat16() for n in lens]
    sink = torch.randn(H, generator=g) if o["sink"] else None
    bias = torch.rand(H, generator=g) if o["bias"] else None
    gates = [torch.randn(n, H, generator=g).bfloat16() if o["gate"] else None for n in lens]
    need = [(len(r) + page - 1) // page for r in rows]
    order, at = torch.randperm(sum(need) + 1, generator=g).tolist(), 0
    cache = torch.full((sum(need) + 1, page, 1, D), float("nan"), dtype=torch.bfloat16)
    table = torch.zeros(len(lens), max(need), dtype=torch.int32)
    for s, r in enumerate(rows):
        for b in range(need[s]):
            piece = r[b * page:(b + 1) * page]
            cache[order[at], :len(piece), 0] = piece
            table[s, b] = order[at]
            at += 1
    dev = "cuda"
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)  # noqa: E731
    out = hip_ops.sink_attention(
        torch.cat(q).to(dev), cache.to(dev), table.to(dev), i32([0] + list(accumulate(lens))), i32([n + c for n, c in zip(lens, ctxs)]), 1, D, C, D ** -0.5,
        max(lens), max(n + c for n, c in zip(lens, ctxs)), sink=sink is not None, sink_logits=None if sink is None else sink.to(dev),
        window_left=o["window"] - 1, keep_first=o["keep"], chunk=o["chunk"], softcap=o["softcap"], value_in_key=True,
        bias_a=None if bias is None else bias.to(dev), bias_b=None if bias is None else torch.full((H,), 0.25, device=dev),
        head_gate=torch.cat(gates).to(dev) if o["gate"] else None).double().cpu()
    at = 0
    for s, n in enumerate(lens):
        ref = reference(q[s].double(), rows[s].double(), C, D ** -0.5, None if sink is None else sink.double(), o["window"], o["keep"], o["chunk"],
                        o["softcap"], None if bias is None else bias.double(), None if gates[s] is None else gates[s].double(), ctxs[s])
        got = out[at:at + n]
        assert torch.isfinite(got).all()
        assert (got - ref).norm() <= BOUND * ref.norm(), (s, float((got - ref).norm() / ref.norm()))
        at += n


@pytest.mark.parametrize("C,H,page,lens,keys", [(256, 8, 64, [1100], 5300), (512, 16, 32, [600, 500], 3000), (256, 3, 16, [1] * 300, 4600), (384, 16, 64, [1] * 270, 4400)])
def test_more_tiles_than_a_look_up_holds(C, H, page, lens, keys):
    """Sequences over the same pages, so many that their keys are not cut: more than 64 tiles one behind the other."""
    from vllm_hymeta import hip_ops
    g, D, T = torch.Generator().manual_seed(C + keys), C + 64, sum(lens)
    rows, q = torch.randn(keys, D, generator=g).bfloat16(), torch.randn(T, H, D, generator=g).bfloat16()
    pages = (keys + page - 1) // page
    order = torch.randperm(pages, generator=g)
    cache = torch.full((pages, page, 1, D), float("nan"), dtype=torch.bfloat16)
    for b in range(pages):
        piece = rows[b * page:(b + 1) * page]
        cache[order[b], :len(piece), 0] = piece
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    out = hip_ops.sink_attention(q.cuda(), cache.cuda(), order.to(torch.int32)[None].expand(len(lens), -1).contiguous().cuda(), i32([0] + list(accumulate(lens))),
                                 i32([keys] * len(lens)), 1, D, C, D ** -0.5, max(lens), keys, value_in_key=True).double().cpu()
    starts = [0] + list(accumulate(lens))
    for s in range(0, len(lens), 1 if len(lens) < 9 else 89):
        some = sorted({0, lens[s] // 2, lens[s] - 1})
        for i in some:                                    # (a row over the keys up to its own)
            n = keys - lens[s] + i + 1
            ref = reference(q[starts[s] + i:starts[s] + i + 1].double(), rows[:n].double(), C, D ** -0.5, None, 0, 0, 0, 0.0, None, None, n - 1)
            got = out[starts[s] + i:starts[s] + i + 1]
            assert (got - ref).norm() <= BOUND * ref.norm(), (s, i)
    assert torch.isfinite(out).all()
