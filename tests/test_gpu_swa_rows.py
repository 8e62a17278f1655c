"""Prefill attention where its blocks of (query, head) rows, its tiles of keys and its copies can go wrong, against the dense
definition in 64 bits."""
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


@pytest.mark.parametrize("page", [16, 48, 64, 192, 256])
@pytest.mark.parametrize("rows,lens,H,G,M,window", [
    ([3, 40, 1], [4500, 100, 64], 7, 1, 0, -1),              # more tiles than a lane table holds; rows over two waves
    ([19, 37], [83, 4300], 14, 2, 32, 200),                  # half a tile of meta keys, a window far into a sequence
    ([129, 65], [129, 1000], 4, 4, 64, 63),                  # one head per key: a block of 128 queries and one more
])
def test_paged_rows(page, rows, lens, H, G, M, window):
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
                                   seq_lens_k=torch.tensor(lens, dtype=torch.int32).cuda(), window_left=window, max_seqlen_k=max(lens),
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
