"""Prefill attention where its blocks of (query, head) rows, its tiles of keys and its copies can go wrong, against the dense
definition in 64 bits."""
import math

import pytest
import torch

from _util import assert_bf16_close, gen, randn_bf16

pytestmark = pytest.mark.gpu
D = 128


def _dense(q, keys, values, ctx, window, meta_k, meta_v):
    """Rows q [n, H, D] behind ``ctx`` of the keys [L, G, D]; meta keys are seen by every row."""
    n, H, G = q.shape[0], q.shape[1], keys.shape[1]
    M = 0 if meta_k is None else meta_k.shape[0]
    if M:
        keys, values = torch.cat((meta_k, keys)), torch.cat((meta_v, values))
    pos, j = torch.arange(ctx, ctx + n)[:, None], torch.arange(keys.shape[0])[None] - M
    seen = (j < 0) | ((j <= pos) & ((window < 0) | (j >= pos - window)))
    k, v = (x.double().repeat_interleave(H // G, 1) for x in (keys, values))
    s = torch.einsum("nhd,lhd->hnl", q.double(), k) * D ** -0.5
    s = s.masked_fill(~seen, -float("inf"))
    p = torch.nan_to_num(torch.softmax(s, -1))               # a row without a key: zero
    return torch.einsum("hnl,lhd->nhd", p, v)


@pytest.mark.parametrize("splits", [0, 1])                    # (by the rule, and one that walks all tiles)
@pytest.mark.parametrize("page", [16, 48, 64, 192, 256])
@pytest.mark.parametrize("rows,lens,H,G,M,window", [
    ([3, 40, 1], [4500, 100, 64], 7, 1, 0, -1),              # more tiles than a lane table holds; rows over two waves
    ([19, 37], [83, 4300], 14, 2, 32, 200),                  # half a tile of meta keys, a window far into a sequence
    ([129, 65], [129, 1000], 4, 4, 64, 63),                  # one head per key: a block of 128 queries and one more
])
def test_paged_rows(page, rows, lens, H, G, M, window, splits):
    from vllm_hymeta import hip_ops

    g_ = gen(3)
    pages = [(n + page - 1) // page for n in lens]
    order = torch.randperm(sum(pages) + 1, generator=g_).tolist()
    table = torch.zeros(len(lens), max(pages), dtype=torch.int32)
    at = 0
    for s, n in enumerate(pages):
        table[s, :n] = torch.tensor(order[at:at + n], dtype=torch.int32)
        at += n
    cache = randn_bf16(g_, 2, sum(pages) + 1, page, G, D)
    live = torch.zeros(sum(pages) + 1, page, dtype=torch.bool)
    q = randn_bf16(g_, sum(rows), H + 1, D)[:, :H]           # (strided rows)
    meta = randn_bf16(g_, 2, M, G, D) if M else None
    cu = torch.tensor([0] + list(torch.tensor(rows).cumsum(0)), dtype=torch.int32)
    want = []
    for s, (r, n) in enumerate(zip(rows, lens)):
        where = table[s, torch.arange(n) // page].long(), torch.arange(n) % page
        live[where] = True
        want.append(_dense(q[cu[s]:cu[s + 1]], cache[0][where], cache[1][where], n - r, window, None if not M else meta[0], None if not M else meta[1]))
    cache[:, ~live] = float("nan")                           # rows behind a sequence's end are nobody's
    kv = cache.cuda()
    out = hip_ops.meta_swa_prefill(q.cuda(), cu.cuda(), max(rows), key_cache=kv[0], value_cache=kv[1], block_tables=table.cuda(),
                                   seq_lens_k=torch.tensor(lens, dtype=torch.int32).cuda(), window_left=window, max_seqlen_k=max(lens), num_splits=splits,
                                   **(dict(meta_key=meta[0].cuda(), meta_value=meta[1].cuda()) if M else {}))
    assert_bf16_close(out.cpu(), torch.cat(want), f"pages of {page}")


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("rows,lens,H,G,M,window", [
    ([70, 0, 9], [40, 5, 9], 6, 2, 0, -1),                   # more queries than keys: the first see nothing; no queries at all
    ([70, 5], [40, 0], 6, 2, 96, 10),                        # ... or the meta keys alone
    ([300], [300], 28, 4, 0, 0),                             # a window of the own key
    ([63, 64, 65, 127, 128, 129], [63, 64, 65, 127, 128, 129], 3, 3, 0, -1),
])
def test_packed_rows(splits, rows, lens, H, G, M, window):
    from vllm_hymeta import hip_ops

    g_ = gen(4)
    q, kv = randn_bf16(g_, sum(rows), H, D), randn_bf16(g_, sum(lens), 2, G, D)
    meta = randn_bf16(g_, 2, M, G, D) if M else None
    cu, ck = (torch.tensor([0] + list(torch.tensor(x).cumsum(0)), dtype=torch.int32) for x in (rows, lens))
    want = [_dense(q[cu[s]:cu[s + 1]], kv[ck[s]:ck[s + 1], 0], kv[ck[s]:ck[s + 1], 1], lens[s] - rows[s], window,
                   None if not M else meta[0], None if not M else meta[1]) for s in range(len(rows))]
    dev = kv.cuda()                                          # (keys and values side by side: rows of 2 G D)
    out = hip_ops.meta_swa_prefill(q.cuda(), cu.cuda(), max(rows), key=dev[:, 0], value=dev[:, 1], cu_seqlens_k=ck.cuda(), window_left=window,
                                   max_seqlen_k=max(lens), num_splits=splits,
                                   **(dict(meta_key=meta[0].cuda(), meta_value=meta[1].cuda()) if M else {}))
    assert_bf16_close(out.cpu(), torch.cat(want), f"{splits} slices")


@pytest.mark.parametrize("splits", [1, 4])
def test_weight_of_the_greatest_score_is_not_rounded(splits):
    """Every row sees one key of weight 1 and one of 3/4, both exact in bf16, beside keys of weights below 2^-40; their values are 1
    and -1, so that an error of the weights' quotient shows 24/7 times as large.  The result, 1/7, is off by its own rounding (2^-9 at most)
    and the scores' errors (fp32: below 2^-18 in the exponent, 2^-16 in the result)."""
    from vllm_hymeta import hip_ops
    n, L, scale = 512, 2048, 2.0 ** -4
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    # scores in base 2: c + 0 and c + log2(3/4) for the two keys, c = 48 .. 56 by row: q = (x, y, 0 ..), keys (1, 0, ..) and (1, 1, 0 ..)
    g = gen(5)
    x = (48 + 8 * torch.rand(n, generator=g)) * math.log(2) / scale
    x = x.bfloat16()
    parts, rest = [], torch.full((n,), math.log(0.75) / scale, dtype=torch.float64)
    for _ in range(3):                                       # log(3/4) in three bf16 parts
        parts.append(rest.bfloat16())
        rest = rest - parts[-1].double()
    q = torch.zeros(n, 1, D).bfloat16()
    q[:, 0, 0] = x
    q[:, 0, 1:4] = torch.stack(parts, 1)
    k, v = torch.zeros(L, 1, D).bfloat16(), torch.zeros(L, 1, D).bfloat16()
    k[5, 0, 0], k[9, 0, :4], v[5], v[9] = 1, 1, 1, -1
    out = hip_ops.meta_swa_prefill(q.cuda(), i32([0, n]), n, key=k.cuda(), value=v.cuda(), cu_seqlens_k=i32([0, L]), scale=scale, num_splits=splits,
                                   max_seqlen_k=L).double().cpu()
    assert (out * 7 - 1).abs().max() < 2.0 ** -9 + 2.0 ** -15


@pytest.mark.parametrize("every", [1, 4])
def test_keys_that_are_not_numbers_stay_in_a_row_of_cut_keys(every):
    """NaN in every tile of the first two of four slices: the row's result is NaN, as where its keys are not cut."""
    from vllm_hymeta import hip_ops
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    q, k, v = (torch.randn(n, h, D, device="cuda").bfloat16() for n, h in ((4, 7), (2048, 1), (2048, 1)))
    k[:1024:every] = float("nan")
    out = hip_ops.meta_swa_prefill(q, i32([0, 4]), 4, key=k, value=v, cu_seqlens_k=i32([0, 2048]), num_splits=4, max_seqlen_k=2048)
    assert out.isnan().all()
