"""The native host side of calls (csrc/calls.cpp) against the same functions in Python: every form that it takes gives the same bytes
and asks for the same room, and what Python refuses is refused with Python's message."""
import pytest
import torch

from _util import gen

pytestmark = pytest.mark.gpu


def _bf(g, *shape):
    return torch.randn(*shape, generator=g).bfloat16().cuda()


def _i32(*values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def _both(monkeypatch, name, call):
    """What ``call`` returns and the rooms it asks for, through the native ``name`` and in Python."""
    from vllm_hymeta import _C, hip_ops
    _C.load()
    module, workspace, found, answered = _C.calls, hip_ops._workspace, [], []
    assert module is not None

    class Counting:
        def __getattr__(self, attribute):
            def native(*args):
                out = getattr(module, attribute)(*args)
                if out is not None:
                    answered.append(attribute)
                return out
            return native
    for calls in (Counting(), None):
        asked = []
        with monkeypatch.context() as m:
            m.setattr(_C, "calls", calls)
            m.setattr(hip_ops, "_workspace", lambda device, nbytes, tag="paged_decode": asked.append((nbytes, tag)) or workspace(device, nbytes, tag))
            found.append(([x.clone() for x in call()], asked))
    (native, rooms), (python, others) = found
    assert answered == [name] and rooms == others
    for x, y in zip(native, python):
        assert x.shape == y.shape and x.dtype == y.dtype and x.stride() == y.stride() and torch.equal(x.view(torch.uint8), y.view(torch.uint8))


SINK = [
    # layout, key and value sizes, heads, key/value heads, rows, contexts, options
    ("rows", 128, 128, 8, 2, [1, 1], [70, 900], dict(sink=True)),
    ("rows", 64, 128, 4, 2, [9, 1, 30], [0, 300, 2000], dict(sink=False, window_left=99, keep_first=5, gate=True)),
    ("rows", 128, 128, 8, 2, [40], [3000], dict(bias=True, softcap=5.0, sink=False)),
    ("rows", 128, 64, 4, 1, [5, 3], [100, 0], dict(chunk=64, sink=False, elem=True)),
    ("latent", 192, 128, 16, 1, [1, 7], [500, 0], dict(sink=True, logits=True)),
    ("latent", 576, 512, 16, 1, [1], [4000], dict(sink=True, logits=True)),
    ("shared", 512, 128, 8, 4, [20], [700], dict(window_left=1023, keep_first=4, sink=False)),
    ("scaled", 128, 128, 8, 2, [3, 1], [300, 40], dict(sink=True, slopes=True, window_left=200)),
    ("rows", 96, 80, 3, 3, [4, 1], [10, 0], dict(sink=False, dtype=torch.float32)),          # the general kernel
]


@pytest.mark.parametrize("layout,D,Dv,H,G,rows,ctx,opts", SINK)
def test_attention_over_paged_rows(monkeypatch, layout, D, Dv, H, G, rows, ctx, opts):
    from vllm_hymeta import hip_ops
    o, g, T, S, page = dict(opts), gen(D + H), sum(rows), len(rows), 64
    dtype = o.pop("dtype", torch.bfloat16)
    lens = [r + c for r, c in zip(rows, ctx)]
    pages = (max(lens) + page - 1) // page
    tail = {"rows": (G, D + Dv), "latent": (1, D), "shared": (1, D + G * Dv), "scaled": (1, hip_ops.scaled_key_row(G, D, dtype))}[layout]
    cache = _bf(g, S * pages, page, *tail).to(dtype)
    q = _bf(g, T, H * D + 8).to(dtype)[:, :H * D].unflatten(1, (H, D))          # (rows further apart than they are long)
    kw = dict(value_in_key=layout == "latent", shared_key=layout == "shared", scaled_key=layout == "scaled")
    if o.pop("gate", False):
        kw["head_gate"] = _bf(g, T, H + 4)[:, :H]
    if o.pop("elem", False):
        kw["elem_gate"] = _bf(g, T, H * Dv)
    if o.pop("bias", False):
        kw.update(bias_a=torch.rand(H, generator=g).cuda(), bias_b=torch.rand(H, generator=g).cuda())
    if o.pop("slopes", False):
        kw["slopes"] = torch.rand(H, generator=g).cuda() * 0.01
    if o.pop("logits", False):
        kw["sink_logits"] = torch.randn(H, generator=g).cuda()
    tables = torch.arange(S * pages, dtype=torch.int32, device="cuda").view(S, pages)
    starts, seq_lens = _i32(*[sum(rows[:i]) for i in range(S + 1)]), _i32(*lens)
    _both(monkeypatch, "sink_attention", lambda: [hip_ops.sink_attention(q, cache, tables, starts, seq_lens, G, D, Dv, D ** -0.5, max(rows), max(lens), **kw, **o)])


@pytest.mark.parametrize("M,window,splits,scale", [(0, -1, 0, None), (32, 99, 0, 0.1), (0, 500, 3, None)])
def test_paged_decode_and_prompts(monkeypatch, M, window, splits, scale):
    from vllm_hymeta import hip_ops
    g, H, G, D, page = gen(M + splits), 8, 2, 128, 16
    cache, tables = _bf(g, 2, 140, page, G, D), torch.arange(140, dtype=torch.int32, device="cuda").view(2, 70)
    meta = dict(meta_key=_bf(g, M, G, D), meta_value=_bf(g, M, G, D)) if M else {}
    kw = dict(window_left=window, num_splits=splits, scale=scale, **meta)
    q = _bf(g, 2, 2 * H, D)[:, :H]
    for longest in (0, 1100):
        _both(monkeypatch, "meta_swa_paged_decode",
              lambda: [hip_ops.meta_swa_paged_decode(q, cache[0], cache[1], _i32(1100, 7), tables, max_seqlen_k=longest, **kw)])
    rows = _bf(g, 40, H, D)
    _both(monkeypatch, "meta_swa_prefill", lambda: [hip_ops.meta_swa_prefill(rows, _i32(0, 33, 40), 33, key_cache=cache[0], value_cache=cache[1], block_tables=tables,
                                                         seq_lens_k=_i32(1100, 7), max_seqlen_k=1100, **kw)])


@pytest.mark.parametrize("rows,D,Dv,dtype", [([1, 1, 1], 128, 128, torch.bfloat16), ([70, 3, 1], 64, 128, torch.bfloat16), ([700], 128, 64, torch.bfloat16),
                                             ([3, 1], 32, 48, torch.float32)])
def test_recurrences(monkeypatch, rows, D, Dv, dtype):
    from vllm_hymeta import hip_ops
    g, H, Hk, T, S = gen(D + Dv), 4, 2, sum(rows), len(rows)
    starts, context, slots = _i32(*[sum(rows[:i]) for i in range(S + 1)]), _i32(*[i % 2 for i in range(S)]), _i32(*[i if i != 1 else -1 for i in range(S)])
    first = torch.randn(S, H, D, Dv, generator=g).cuda()
    rows_of = _bf(g, T, 2 * Hk * D + H * Dv).to(dtype)
    q, k, v = (x.unflatten(1, (n, -1)) for x, n in zip(rows_of.split([Hk * D, Hk * D, H * Dv], 1), (Hk, Hk, H)))
    qkv, decay, log2 = _bf(g, T, H * (2 * D + Dv)).to(dtype), (torch.rand(H, generator=g) * 0.2 + 0.8).cuda(), (-torch.rand(T, H, generator=g)).cuda()
    scale, skip, beta = torch.rand(T, H, generator=g).cuda(), torch.randn(H, generator=g).cuda(), _bf(g, T, H + 3).to(dtype)[:, :H]
    where = (starts, context, slots, max(rows))

    def with_state(name, call):
        def run():
            state = first.clone()
            return [call(state), state]
        _both(monkeypatch, name, run)
    with_state("lightning_attention", lambda s: hip_ops.lightning_attention(qkv, s, decay, H, D, Dv, *where))
    with_state("decay_scan", lambda s: hip_ops.decay_scan(q, k, v, s, *where, decay=decay))
    with_state("decay_scan", lambda s: hip_ops.decay_scan(q, k, v, s, *where, log2_decay=log2, v_scale=scale, skip=skip))
    with_state("delta_rule", lambda s: hip_ops.delta_rule(q, k, v, beta, log2, s, *where, D ** -0.5, 1e-6))


def test_refused_as_in_python(monkeypatch):
    from vllm_hymeta import _C, hip_ops
    _C.load()
    g = gen(3)
    q, cache, tables = _bf(g, 2, 4, 128), _bf(g, 4, 64, 2, 256), torch.zeros(2, 2, dtype=torch.int32, device="cuda")
    starts, lens, state, slots = _i32(0, 1, 2), _i32(70, 3), torch.zeros(2, 4, 128, 128, device="cuda"), _i32(0, 1)
    sink = lambda **kw: hip_ops.sink_attention(*[kw.pop(n, x) for n, x in (("q", q), ("cache", cache), ("tables", tables), ("starts", starts), ("lens", lens))],  # noqa: E731
                                               2, 128, 128, 0.1, 1, 70, **kw)
    scan = lambda **kw: hip_ops.decay_scan(*[kw.pop(n, x) for n, x in (("q", q), ("k", q), ("v", q), ("state", state))], starts, slots, slots, 1, **kw)  # noqa: E731
    decay = torch.ones(4, device="cuda")
    wrong = [lambda: sink(q=q.half()), lambda: sink(cache=cache.float()), lambda: sink(cache=cache[:, ::2]), lambda: sink(tables=tables.long()), lambda: sink(lens=lens.cpu()),
             lambda: sink(lens=lens.long()), lambda: sink(chunk=4, window_left=3), lambda: sink(slopes=decay, bias_a=decay, bias_b=decay), lambda: sink(bias_a=decay),
             lambda: sink(q=q.transpose(1, 2)), lambda: sink(sink_logits=decay[:2]), lambda: sink(head_gate=q[:, :, 0].float()), lambda: sink(value_in_key=True, shared_key=True),
             lambda: scan(), lambda: scan(decay=decay, log2_decay=torch.zeros(2, 4, device="cuda")), lambda: scan(decay=decay.bfloat16()), lambda: scan(decay=decay, state=state.bfloat16()),
             lambda: scan(decay=decay, state=state[:, :, ::2]), lambda: scan(decay=decay, k=q.float()), lambda: scan(decay=decay, v=q[:1]),
             lambda: hip_ops.meta_swa_paged_decode(q, cache[..., :128], cache[..., 128:].contiguous(), lens, tables)]
    for call in wrong:
        messages = []
        for calls in (_C.calls, None):
            with monkeypatch.context() as m, pytest.raises((ValueError, _C.HymetaError)) as error:
                m.setattr(_C, "calls", calls)
                call()
            messages.append((type(error.value), str(error.value)))
        assert messages[0] == messages[1]


def _long_prompt(hip_ops, rows=700, **kw):
    g = gen(rows)
    qkv, state, decay = _bf(g, rows, 4 * 384), torch.zeros(1, 4, 128, 128, device="cuda"), torch.full((4,), 0.9, device="cuda")
    return hip_ops.lightning_attention(qkv, state, decay, 4, 128, 128, _i32(0, rows), _i32(0), _i32(0), kw.get("most", rows))


@pytest.mark.parametrize("error", [KeyboardInterrupt, RuntimeError, torch.cuda.OutOfMemoryError])
def test_an_exception_in_between_is_the_calls(monkeypatch, error):
    """What is raised while the native side asks for a workspace is not taken for a refusal."""
    from vllm_hymeta import _C, hip_ops
    _C.load()
    workspace, raised = hip_ops._workspace, []

    def once(*args):
        if not raised:
            raised.append(args)
            raise error("in between")
        return workspace(*args)
    monkeypatch.setattr(hip_ops, "_workspace", once)
    with pytest.raises(error, match="in between"):
        _long_prompt(hip_ops)
    assert len(raised) == 1 and torch.isfinite(_long_prompt(hip_ops)).all()


def _small_calls(hip_ops):
    """Name and call of one small problem of every function but the recurrences' siblings."""
    g = gen(11)
    q, cache, tables = _bf(g, 2, 4, 128), _bf(g, 2, 8, 64, 2, 128), torch.arange(8, dtype=torch.int32, device="cuda").view(2, 4)
    rows, starts, lens, slots = _bf(g, 2, 4 * 384), _i32(0, 1, 2), _i32(130, 3), _i32(0, 1)
    state, log2, decay = torch.zeros(2, 4, 128, 128, device="cuda"), torch.zeros(2, 4, device="cuda"), torch.full((4,), 0.9, device="cuda")
    both = _bf(g, 8, 64, 2, 256)
    return [
        ("sink_attention", lambda: hip_ops.sink_attention(q, both, tables, starts, lens, 2, 128, 128, 0.1, 1, 130)),
        ("meta_swa_paged_decode", lambda: hip_ops.meta_swa_paged_decode(q, cache[0], cache[1], lens, tables)),
        ("meta_swa_prefill", lambda: hip_ops.meta_swa_prefill(q, starts, 1, key_cache=cache[0], value_cache=cache[1], block_tables=tables, seq_lens_k=lens, max_seqlen_k=130)),
        ("lightning_attention", lambda: hip_ops.lightning_attention(rows, state.clone(), decay, 4, 128, 128, starts, lens, slots, 1)),
        ("decay_scan", lambda: hip_ops.decay_scan(q, q, q, state.clone(), starts, lens, slots, 1, decay=decay)),
        ("delta_rule", lambda: hip_ops.delta_rule(q, q, q, q[:, :, 0].contiguous(), log2, state.clone(), starts, lens, slots, 1, 0.1, 1e-6)),
    ]


@pytest.mark.parametrize("at", range(6))
def test_outputs_come_from_what_stands_for_torch_empty(monkeypatch, at):
    from vllm_hymeta import _C, hip_ops
    _C.load()
    name, call = _small_calls(hip_ops)[at]
    call()                                                   # (its workspace is there)
    plain, empty, made, module, answered = call(), torch.empty, [], _C.calls, []

    class Noting:
        def __getattr__(self, attribute):
            return lambda *args: answered.append(attribute) or getattr(module, attribute)(*args)

    def filled(*size, **kw):
        made.append(empty(*size, **kw).fill_(7))
        return made[-1]
    monkeypatch.setattr(_C, "calls", Noting())
    monkeypatch.setattr(torch, "empty", filled)
    out = call()
    assert answered == [name] and len(made) == 1 and made[0].data_ptr() == out.data_ptr() and torch.equal(out, plain)


@pytest.mark.parametrize("at", range(6))
def test_on_another_stream_and_inside_a_mode(monkeypatch, at):
    from torch.utils._python_dispatch import TorchDispatchMode
    from vllm_hymeta import hip_ops
    name, call = _small_calls(hip_ops)[at]
    plain, side = call(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _both(monkeypatch, name, lambda: [call()])
    torch.cuda.current_stream().wait_stream(side)

    class Through(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    with Through():
        inside = call()
    assert torch.equal(inside, plain)


def test_subclasses_and_transforms_are_left_to_python(monkeypatch):
    from vllm_hymeta import _C, hip_ops
    _C.load()

    class Own(torch.Tensor):
        pass
    g = gen(5)
    rows, starts, lens, slots, decay = _bf(g, 2, 4 * 384), _i32(0, 1, 2), _i32(0, 3), _i32(0, 1), torch.full((4,), 0.9, device="cuda")
    state = torch.zeros(2, 4, 128, 128, device="cuda")
    run = lambda x: hip_ops.lightning_attention(x, state.clone(), decay, 4, 128, 128, starts, lens, slots, 1)  # noqa: E731
    args = (decay, 4, 128, 128, state.clone(), starts, lens, slots, 1, torch.cuda.current_stream().cuda_stream)
    assert _C.calls.lightning_attention(rows.as_subclass(Own), *args) is None
    assert torch.equal(run(rows.as_subclass(Own)).as_subclass(torch.Tensor), run(rows))
    errors = []
    for calls in (_C.calls, None):
        with monkeypatch.context() as m, pytest.raises(RuntimeError) as error:
            m.setattr(_C, "calls", calls)
            torch.vmap(run)(rows[None].expand(3, -1, -1))
        errors.append(str(error.value))
    assert errors[0] == errors[1]
