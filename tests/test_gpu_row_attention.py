"""Prompts' portions of the paged attention, keys of 32 to 192 elements in every layout of a cache row, at the edges of the
kernel's tiles: 32 (query, head) rows a wave and 128 a workgroup, 64 keys a tile, pages that hold a tile and pages that do not,
and portions short enough that their keys are cut into slices (2 tiles a slice or more).

Bound: the outputs are bf16 (2^-9 of each value at most); the weights are two bf16 parts (2^-17), exponentials, logarithms and
products fp32 (below 2^-11 over these lengths and biases); together below 2^-9 + 2^-10 in the norm."""
from itertools import accumulate

import pytest
import torch

pytestmark = pytest.mark.gpu
BOUND = 2.0 ** -9 + 2.0 ** -10
SLOPE, NEAR = 0.03, 0.25


def reference(q, k, v, scale, ctx, o, sink, a, gate):
    """One sequence in 64 bits: q [n, H, D] at positions ctx .., k [H, ctx + n, D], v [H, ctx + n, Dv]."""
    n = q.shape[0]
    i, j = torch.arange(ctx, ctx + n)[:, None], torch.arange(ctx + n)
    seen = j <= i
    if o["chunk"]:
        seen = seen & (j >= i // o["chunk"] * o["chunk"])
    elif o["window"]:
        seen = seen & ((j > i - o["window"]) | (j < o["keep"]))
    s = torch.einsum("nhd,hjd->hnj", q, k) * scale
    if o["softcap"]:
        s = o["softcap"] * torch.tanh(s / o["softcap"])
    far = (i - j).clamp_min(0).double()
    if o["bias"] == "log":
        s = s - a[:, None, None] * torch.log1p(o["near"] * far)
    elif o["bias"] == "linear":
        s = s - SLOPE * a[:, None, None] * far
    s = s.masked_fill(~seen, float("-inf"))
    if sink is not None:
        s = torch.cat((s, sink[:, None, None].expand(len(sink), n, 1)), -1)
    out = torch.einsum("hnj,hjc->nhc", torch.softmax(s, -1)[..., :ctx + n].nan_to_num(), v)      # (no keys: 0)
    return out if gate is None else out * torch.sigmoid(gate)[:, :, None]


@pytest.mark.parametrize("layout,D,Dv,H,G,page,lens,ctxs,opts", [
    ("rows", 128, 128, 28, 4, 64, [18, 2, 19], [0, 64, 700], dict(sink=True, bias="log")),       # 126, 14 and 133 rows
    ("rows", 128, 64, 4, 1, 16, [32, 33, 1], [31, 0, 70], dict(softcap=4.0)),                    # small pages
    ("rows", 64, 128, 2, 2, 64, [129, 64], [1, 512], dict(window=70, keep=9)),                   # one head a key/value head, kept keys
    ("rows", 64, 64, 6, 2, 128, [5, 3], [1000, 2000], dict(chunk=300, gate=True)),
    ("rows", 128, 128, 8, 2, 64, [3, 2], [3000, 63], dict(softcap=6.0, bias="log", sink=True)),  # slices, of which some see nothing
    ("rows", 128, 128, 8, 2, 64, [70, 3], [200, 0], dict(sink=True, bias="log", near=98765.43)),     # steep biases: the nearest keys'
    ("rows", 128, 128, 8, 2, 64, [70, 3], [200, 0], dict(sink=True, bias="log", near=987654.3)),     # logarithms from exact distances
    ("latent", 192, 128, 8, 1, 64, [33, 3], [100, 0], dict(sink=True, bias="log", near=98765.43)),
    ("rows", 128, 128, 4, 2, 64, [3, 200, 1, 2], [-1, -150, -1, -2], {}),                        # rows in front of their sequence
    ("rows", 64, 64, 4, 2, 16, [3, 70, 1], [-2, -30, -1], dict(chunk=20)),
    ("scaled", 64, 64, 4, 2, 64, [2, 70, 1], [-1, -30, 3000], dict(sink=True, window=30)),
    ("latent", 192, 128, 16, 1, 64, [8, 9, 2], [0, 63, 1500], dict(sink=True)),
    ("latent", 160, 128, 5, 1, 32, [70], [11], dict(bias="log")),
    ("latent", 128, 64, 3, 1, 64, [90, 2], [0, 900], dict(window=200)),
    ("latent", 96, 64, 7, 1, 8, [40, 64], [5, 64], dict(sink=True)),
    ("shared", 128, 64, 4, 2, 64, [50, 2], [14, 800], dict(window=100, keep=4)),
    ("shared", 64, 128, 4, 4, 64, [65], [64], {}),
    # keys cut into slices: a window with kept first keys and both gates, beside single rows, some blocks cut and some whole
    ("rows", 128, 128, 8, 2, 64, [40, 1, 1, 3, 1], [3000, 900, 64, 10, 2000], dict(window=2100, keep=70, gate=True, elem=True)),
    ("rows", 64, 64, 4, 2, 16, [1, 9, 1], [70, 2500, 1300], dict(window=1500, keep=9, elem=True, sink=True)),
    ("rows", 128, 64, 6, 2, 64, [5, 1, 50], [2900, 100, 0], dict(chunk=1000, gate=True, elem=True)),
    ("latent", 192, 128, 40, 1, 64, [7, 1, 4], [2000, 1500, 0], dict(elem=True, gate=True)),      # two launches of heads for single rows
    ("scaled", 64, 64, 4, 2, 64, [3, 1, 17], [2500, 3000, 600], dict(sink=True, bias="linear", window=2000, keep=5, elem=True)),
    ("scaled", 128, 128, 28, 4, 64, [20, 2], [0, 1200], dict(sink=True, bias="linear")),
    ("scaled", 96, 96, 4, 2, 16, [33, 70], [100, 0], dict(bias="linear", window=50)),
    ("scaled", 64, 64, 4, 1, 64, [64], [64], dict(sink=True)),
    ("scaled", 32, 32, 3, 3, 64, [10, 11], [700, 0], dict(bias="linear")),
    # the shortest keys that are cut: 3, 4 and 5 tiles
    *[("rows", 128, 128, 8, 2, 64, [8, 2], [c, 63], dict(sink=True, gate=True)) for c in (184, 185, 248, 249)],
    # single rows: as many partials as a thread of the merge holds, and one more; head groups that are not full
    *[("rows", 64, 64, 10, 2, 64, [1, 0, 1, 1], [64 * n - 1, 5, 0, 70], dict(sink=True, gate=True, elem=True)) for n in (2, 3, 4, 5, 8, 9)],
    # and as many as its threads take at once, four or eight each, and one more; statistics for two each
    *[("rows", 64, 64, 10, 2, 64, [1], [64 * n - 1], dict(sink=True, gate=True, elem=True)) for n in (32, 33, 64, 65, 129)],
    ("rows", 64, 128, 3, 1, 64, [1, 1], [63, -1], {}),
    ("latent", 192, 128, 37, 1, 64, [1, 1], [127, 3], dict(sink=True, elem=True)),
    ("scaled", 96, 96, 7, 7, 64, [1, 1], [200, 3], dict(sink=True, bias="linear")),
    # few keys: single rows among the portions' blocks, up to the last such length and one key past it
    *[("rows", 128, 128, 28, 4, 64, [1, 5, 0, 1, 40, 1], [0, 3, 0, c, 100, -1], dict(sink=True, bias="log", gate=True)) for c in (1023, 1024)],
    ("latent", 192, 128, 16, 1, 64, [1, 1, 9], [511, 63, 0], dict(sink=True, elem=True)),
    ("scaled", 64, 64, 4, 2, 64, [1, 2, 1], [700, 30, 5000], dict(sink=True, bias="linear", window=500, keep=7)),
    ("shared", 128, 64, 4, 2, 16, [3, 1], [100, 255], {}),
    # keys cut into slices beside more single rows than go among the portions' blocks
    ("rows", 64, 64, 4, 2, 64, [9] + [1] * 40, [2500] + [31 * i for i in range(40)], dict(sink=True, gate=True)),
    ("latent", 192, 128, 8, 1, 64, [30] + [1] * 70, [1500] + [17 * i for i in range(70)], {}),
])
def test_against_64_bits(layout, D, Dv, H, G, page, lens, ctxs, opts):
    from vllm_hymeta import hip_ops
    dev, g = "cuda", torch.Generator().manual_seed(D + H)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)  # noqa: E731
    o = dict(dict(sink=False, window=0, keep=0, chunk=0, softcap=0.0, bias=None, gate=False, elem=False, near=NEAR), **opts)
    key_heads = 1 if layout in ("latent", "shared") else G
    total = [n + c for n, c in zip(lens, ctxs)]
    keys = [torch.randn(t, key_heads, D, generator=g).bfloat16() for t in total]
    values = [k[:, :, :Dv] if layout in ("latent", "scaled") else torch.randn(len(k), G, Dv, generator=g).bfloat16() for k in keys]
    q = [torch.randn(n, H, D, generator=g).bfloat16() for n in lens]
    sink = torch.randn(H, generator=g) if o["sink"] else None
    a = 0.1 + torch.rand(H, generator=g)
    gates = [torch.randn(n, H, generator=g).bfloat16() if o["gate"] else None for n in lens]
    elems = [torch.randn(n, H * Dv, generator=g).bfloat16() if o["elem"] else None for n in lens]
    need = [(t + page - 1) // page for t in total]
    order, at = torch.randperm(sum(need) + 1, generator=g).tolist(), 0
    tail = {"rows": (G, D + Dv), "latent": (1, D), "shared": (1, D + G * Dv), "scaled": (1, hip_ops.scaled_key_row(G, D, torch.bfloat16))}[layout]
    cache = torch.full((sum(need) + 1, page) + tail, float("nan"), dtype=torch.bfloat16, device=dev)
    table = torch.zeros(len(lens), max(need), dtype=torch.int32)
    for s in range(len(lens)):
        pages = order[at:at + need[s]]
        at += need[s]
        table[s, :need[s]] = torch.tensor(pages, dtype=torch.int32)
        slots = torch.tensor([pages[p // page] * page + p % page for p in range(total[s])], dtype=torch.int64, device=dev)
        if layout == "scaled":
            qk = torch.cat((torch.zeros(total[s], D).bfloat16(), keys[s].reshape(total[s], -1)), 1).to(dev)
            ones = torch.ones(D, device=dev)
            hip_ops.scaled_key_cache_(qk, 1, G, D, ones, ones, 1e-6, cache, slots)
            continue
        row = {"rows": lambda: torch.cat((keys[s], values[s]), 2), "latent": lambda: keys[s],
               "shared": lambda: torch.cat((keys[s].reshape(total[s], 1, D), values[s].reshape(total[s], 1, -1)), 2)}[layout]()
        cache.view((-1,) + tail)[slots] = row.to(dev)
    out = hip_ops.sink_attention(
        torch.cat(q).to(dev), cache, table.to(dev), i32([0] + list(accumulate(lens))), i32(total), G if layout != "latent" else 1, D, Dv, D ** -0.5,
        max(lens), max(total), sink=sink is not None, sink_logits=None if sink is None else sink.to(dev), window_left=o["window"] - 1,
        keep_first=o["keep"], chunk=o["chunk"], softcap=o["softcap"], value_in_key=layout == "latent", shared_key=layout == "shared",
        scaled_key=layout == "scaled", bias_a=a.to(dev) if o["bias"] == "log" else None, slopes=(SLOPE * a).to(dev) if o["bias"] == "linear" else None,
        bias_b=torch.full((H,), o["near"], device=dev) if o["bias"] == "log" else None,
        head_gate=torch.cat(gates).to(dev) if o["gate"] else None, elem_gate=torch.cat(elems).to(dev) if o["elem"] else None).double().cpu()
    at = 0
    for s, n in enumerate(lens):
        k, v = keys[s].double(), values[s].double()
        if layout == "scaled":
            k = k * torch.rsqrt(k.square().mean(-1, keepdim=True) + 1e-6)
        spread = lambda x: x.permute(1, 0, 2).repeat_interleave(H // x.shape[1], 0)  # noqa: E731
        ref = reference(q[s].double(), spread(k), spread(v), D ** -0.5, ctxs[s], o, None if sink is None else sink.double(), a.double(),
                        None if gates[s] is None else gates[s].double())
        if elems[s] is not None:
            ref = ref * torch.sigmoid(elems[s].double()).reshape(ref.shape)
        got = out[at:at + n]
        assert torch.isfinite(got).all()
        assert (got - ref).norm() <= BOUND * ref.norm(), (s, float((got - ref).norm() / ref.norm()))
        at += n


@pytest.mark.parametrize("D,Dv", [(128, 128), (576, 512)])
def test_rows_behind_the_last_portion_stay_untouched(D, Dv, monkeypatch):
    """Six rows more than the portions have, with keys cut into slices: nothing is written for them."""
    from vllm_hymeta import hip_ops
    dev = "cuda"
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)  # noqa: E731
    inside, empty = D != Dv, torch.empty
    q, cache = torch.randn(11, 4, D, device=dev).bfloat16(), torch.randn(32, 64, 1, D if inside else D + Dv, device=dev).bfloat16()
    monkeypatch.setattr(torch, "empty", lambda *size, **kw: empty(*size, **kw).fill_(7))
    out = hip_ops.sink_attention(q, cache, torch.arange(32, dtype=torch.int32, device=dev)[None], i32([0, 5]), i32([2048]), 1, D, Dv, D ** -0.5, 5, 2048,
                                 value_in_key=inside)
    assert (out[5:] == 7).all() and torch.isfinite(out).all() and not (out[:5] == 7).all()


@pytest.mark.parametrize("D,Dv", [(128, 128), (576, 512)])
@pytest.mark.parametrize("lens", [[1], [0, 2], [1, 0, 1]])
def test_bounds_larger_than_the_step(D, Dv, lens):
    """The step's lengths are bounds: fewer rows than the longest portion may have, and sequences without rows."""
    from vllm_hymeta import hip_ops
    dev, T = "cuda", sum(lens)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)  # noqa: E731
    inside = D != Dv
    q, cache = torch.randn(T, 4, D, device=dev).bfloat16(), torch.randn(8, 64, 1, D if inside else D + Dv, device=dev).bfloat16()
    table = torch.arange(8, dtype=torch.int32, device=dev)[None].repeat(len(lens), 1)
    starts, ends = i32([0] + list(accumulate(lens))), i32([300 + n for n in lens])
    run = lambda most_rows, most_keys: hip_ops.sink_attention(q, cache, table, starts, ends, 1, D, Dv, D ** -0.5, most_rows, most_keys, value_in_key=inside)  # noqa: E731
    a, b = run(max(lens), 300 + max(lens)).double(), run(500, 512).double()
    assert torch.isfinite(a).all() and (a - b).norm() <= BOUND * a.norm()


@pytest.mark.parametrize("D,dtype", [(512, torch.bfloat16), (128, torch.float32)])
def test_kernels_without_slices_ask_for_no_room_for_them(D, dtype, monkeypatch):
    from vllm_hymeta import _C, hip_ops
    dev, asked, workspace = "cuda", [], hip_ops._workspace
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)  # noqa: E731
    monkeypatch.setattr(hip_ops, "_workspace", lambda device, nbytes, tag: asked.append(nbytes) or workspace(device, nbytes, tag))
    q, cache = torch.randn(5, 4, D, device=dev).to(dtype), torch.randn(64, 64, 1, D + 2 * 64, device=dev).to(dtype)
    out = hip_ops.sink_attention(q, cache, torch.arange(64, dtype=torch.int32, device=dev)[None], i32([0, 5]), i32([4096]), 2, D, 64, D ** -0.5, 5, 4096, shared_key=True)
    assert asked == [_C.load().hymeta_sink_attention_workspace_bytes(1, 4, 2, 64, 4096)] and torch.isfinite(out).all()


@pytest.mark.parametrize("layout,D,Dv,H,G,rows,ctx,scale,opts", [
    ("rows", 64, 128, 8, 8, 4300, 0, 0.125, dict(sink=True, bias=True)),          # more tiles than a lane table holds
    ("rows", 128, 64, 14, 2, 2500, 2100, -0.08, dict(keep=9, window=2200)),       # scores that fall with their products
    ("rows", 128, 128, 4, 4, 4500, 1, 0.1, dict(softcap=3.0, chunk=4300)),
    ("shared", 64, 64, 6, 6, 4400, 77, 0.125, dict(sink=True)),
])
def test_long_portions_against_the_general_kernel(layout, D, Dv, H, G, rows, ctx, scale, opts):
    """Pages of 64 against pages of 48, which only the kernel of one row per wave reads."""
    from vllm_hymeta import hip_ops
    dev, g, total = "cuda", torch.Generator().manual_seed(D + rows), rows + ctx
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)  # noqa: E731
    tail = (1, D + G * Dv) if layout == "shared" else (G, D + Dv)
    keys, q = torch.randn((total,) + tail, generator=g).bfloat16().to(dev), torch.randn(rows, H, D, generator=g).bfloat16().to(dev)
    bias = dict(bias_a=(0.1 + torch.rand(H, generator=g)).to(dev), bias_b=torch.full((H,), NEAR, device=dev)) if opts.get("bias") else {}
    outs = []
    for page in (64, 48):
        pages = (total + page - 1) // page
        table = torch.randperm(pages, generator=g).to(torch.int32).to(dev)
        cache = torch.full((pages * page,) + tail, float("nan"), dtype=torch.bfloat16, device=dev)
        j = torch.arange(total, device=dev)
        cache[table[j // page].long() * page + j % page] = keys
        outs.append(hip_ops.sink_attention(q, cache.view((pages, page) + tail), table[None], i32([0, rows]), i32([total]), G, D, Dv, scale, rows, total,
                                           sink=opts.get("sink", False), softcap=opts.get("softcap", 0.0), chunk=opts.get("chunk", 0),
                                           window_left=opts.get("window", 0) - 1, keep_first=opts.get("keep", 0), shared_key=layout == "shared", **bias).double())
    assert all(torch.isfinite(o).all() for o in outs)
    assert (outs[0] - outs[1]).norm() <= 2 * BOUND * outs[1].norm()             # (each within BOUND of the exact result)


@pytest.mark.parametrize("D,Dv,lens", [(128, 128, [4]), (192, 128, [4]), (576, 512, [4]), (128, 128, [1]), (576, 512, [1])])
@pytest.mark.parametrize("every", [1, 4])
def test_keys_that_are_not_numbers_stay_in_a_row_of_cut_keys(D, Dv, lens, every):
    """NaN in every tile of the first 1536 keys, where slices of 2, 3 and 4 tiles of 64 end, so that none sees both kinds: the row's
    result is NaN, as where its keys are not cut."""
    from vllm_hymeta import hip_ops
    dev, total = "cuda", 3000
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)  # noqa: E731
    inside = D != Dv
    q, cache = torch.randn(sum(lens), 4, D, device=dev).bfloat16(), torch.randn(47, 64, 1, D if inside else D + Dv, device=dev).bfloat16()
    cache.view(-1, cache.shape[-1])[:1536:every, :64] = float("nan")           # (of a key alone; where it holds the value, of that too)
    out = hip_ops.sink_attention(q, cache, torch.arange(47, dtype=torch.int32, device=dev)[None], i32([0] + list(accumulate(lens))), i32([total]), 1, D, Dv,
                                 D ** -0.5, max(lens), total, value_in_key=inside)
    assert out.isnan().all()


@pytest.mark.parametrize("layout", ["rows", "shared"])
@pytest.mark.parametrize("opts", [{}, dict(softcap=5.0), dict(window_left=20)])
def test_scale_of_zero_weighs_all_keys_alike(layout, opts):
    """Scores of 0: a row is the mean of the values it sees."""
    from vllm_hymeta import hip_ops
    dev, n, D = "cuda", 100, 128
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)  # noqa: E731
    q, cache = torch.randn(n, 4, D, device=dev).bfloat16(), torch.randn(2, 64, 1, 2 * D, device=dev).bfloat16()
    out = hip_ops.sink_attention(q, cache, i32([[0, 1]]), i32([0, n]), i32([n]), 1, D, D, 0.0, n, n, sink=False,
                                 shared_key=layout == "shared", **opts).double()
    i = torch.arange(n, device=dev)
    seen = ((i[None] <= i[:, None]) & (i[None] >= i[:, None] - opts.get("window_left", n))).double()
    want = (seen @ cache.view(-1, 2 * D)[:n, D:].double() / seen.sum(1, keepdim=True))[:, None].expand(n, 4, D)
    assert (out - want).norm() <= BOUND * want.norm()
