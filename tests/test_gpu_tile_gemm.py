"""The tiled matrix products of prompts (256 x 256 tiles, halves of 128 rows), bit for bit: operands are small integers and
scales powers of two, so that every fp32 sum is exact in any order and one rounding to bf16 remains."""
import ctypes as C

import pytest
import torch

from _util import gen

pytestmark = pytest.mark.gpu

NONE, SILU, SILU_EXACT, CLAMPED = 0, 1, 2, 3


def _ints(g, lo, hi, *shape):
    return torch.randint(lo, hi + 1, shape, generator=g)


def _activate(h, act):
    from vllm_hymeta import hip_ops
    if act == NONE:
        return h
    if act == SILU:
        return hip_ops.silu_and_mul(h)
    return hip_ops.silu_mul(h) if act == SILU_EXACT else hip_ops.clamped_glu(h, 7.0, 1.702)


@pytest.mark.parametrize("sizes,K,N,div,local,act,int8", [
    # rows at the edges of tiles and halves, an expert without rows; the fewest steps; more than a round of tiles
    ((1, 255, 256, 257, 0, 511, 129, 128), 256, 10240, 1, (0, 8), NONE, False),
    ((1, 255, 256, 257, 0, 511, 129, 128), 320, 10240, 2, (0, 8), SILU, False),      # an odd number of steps; two slots a source row
    ((700, 3, 1100), 256, 8704, 1, (0, 3), CLAMPED, False),                          # a last round of at most half the units: halves
    ((700, 3, 1100), 512, 5120, 1, (0, 3), SILU_EXACT, False),
    ((640, 333, 200, 515), 512, 5120, 1, (1, 3), SILU, True),                        # a rank's share of the experts
    ((1, 255, 256, 257, 0, 511, 129, 128), 640, 10240, 2, (0, 8), NONE, True),
    ((2600,), 1024, 5120, 1, (0, 1), NONE, True),                                    # more row tiles than a block of neighbours holds
    ((5, 900), 256, 10240, 1, (0, 1), SILU, False),                                  # halves that hold no rows
    ((2600, 1300), 448, 2560, 3, (0, 2), NONE, False),
    ((8500, 3, 700), 256, 1280, 1, (0, 3), NONE, False),                             # more row tiles than the columns are swept once for
    ((16640, 300), 512, 1536, 1, (0, 2), SILU, True),                                # three sweeps of one expert, the last of one row tile
    ((128, 140, 0, 126, 150, 257, 1, 250) * 8, 256, 1024, 1, (0, 64), NONE, False),  # an expert for every lane
    ((128, 140, 0, 126, 150, 257, 1, 250) * 8, 512, 1024, 2, (3, 61), SILU, True),
])
def test_grouped_products(sizes, K, N, div, local, act, int8):
    from vllm_hymeta import _C
    lib, E, P = _C.load(), len(sizes), sum(sizes)
    g = gen(7)
    kind = torch.int8 if int8 else torch.bfloat16
    T = (P + div - 1) // div
    x, w = _ints(g, -3, 3, T, K), _ints(g, -2, 2, E, N, K)
    slots = torch.randperm(T * div, generator=g)[:P]
    factor = 2.0 ** _ints(g, -2, 1, P).float()
    order = torch.randperm(P, generator=g)
    offsets = torch.tensor([0] + list(sizes)).cumsum(0)
    x_scale, w_scale = 2.0 ** _ints(g, -3, 0, T).float(), 2.0 ** _ints(g, -2, 1, E, N).float()
    d = {n: t.cuda() for n, t in dict(x=x.to(kind), w=w.to(kind), slots=slots.int(), factor=factor, order=order.int(),
                                      offsets=offsets.int(), x_scale=x_scale, w_scale=w_scale).items()}
    cols = N // 2 if act else N
    out = torch.full((P + 1, cols), 7.0, dtype=torch.bfloat16, device="cuda")
    a = _C.MoeGemmArgs()
    ptr = lambda t: C.c_void_p(t.data_ptr())      # noqa: E731
    a.x, a.weights, a.out, a.expert_offsets = ptr(d["x"]), ptr(d["w"]), ptr(out), ptr(d["offsets"])
    a.a_rows, a.a_rows_div, a.scale_rows, a.row_scale = ptr(d["slots"]), div, ptr(d["order"]), ptr(d["factor"])
    a.max_rows, a.K, a.N = P, K, N
    a.local_expert_begin, a.local_expert_end = local
    a.x_stride_m, a.out_stride_m, a.w_stride_e = K, cols, N * K
    if int8:
        a.operand_dtype, a.x_scale, a.w_scale = _C.HYMETA_I8, ptr(d["x_scale"]), ptr(d["w_scale"])
    assert lib.hymeta_moe_gemm_activates(C.byref(a)) == 1            # these sizes are the tiles'
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    if act:
        assert lib.hymeta_moe_gemm_act(C.byref(a), act, 7.0, 1.702, stream) == 0
    else:
        assert lib.hymeta_moe_gemm(C.byref(a), stream) == 0
    torch.cuda.synchronize()
    source = slots // div
    for e in range(E):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        if not local[0] <= e < local[1]:
            assert bool((out[lo:hi] == 7.0).all())                   # other ranks' rows stay as they are
            continue
        if lo == hi:
            continue
        s = source[lo:hi].cuda()
        h = d["x"][s].float() @ d["w"][e].float().t()                # exact: |sums| < 2^24
        if int8:
            h = h * d["x_scale"][s][:, None] * d["w_scale"][e]
        h = (h * d["factor"][d["order"][lo:hi].long()][:, None]).to(torch.bfloat16)
        assert torch.equal(out[lo:hi], _activate(h, act)), f"expert {e}"
    assert bool((out[P] == 7.0).all())


@pytest.mark.parametrize("sizes,K,N,local,total", [
    ((1, 255, 256, 257, 0, 511, 129, 200), 2048, 5120, (0, 8), 0),               # 201 rows an expert on average, tiles of eight waves
    ((200, 140, 160, 141) * 2, 2080, 5120, (0, 8), 0),                           # 160; an odd number of steps
    ((239,) * 8, 2048, 5120, (0, 8), 0),
    ((200, 3, 0, 260, 130, 190, 300, 129, 17), 2112, 5376, (1, 9), 9),           # eight of nine
    ((20, 80, 0, 300, 75, 129, 5, 64) * 2, 256, 10240, (8, 16), 16),             # a rank's half of 1346 pairs: 84 rows an expert, tiles of 128
])
def test_grouped_products_by_the_rows_of_an_expert(sizes, K, N, local, total):
    from vllm_hymeta import _C
    lib, E, P = _C.load(), len(sizes), sum(sizes)
    g = gen(23)
    x, w = _ints(g, -3, 3, P, K).bfloat16().cuda(), _ints(g, -2, 2, E, N, K).bfloat16().cuda()
    offsets = torch.tensor([0] + list(sizes)).cumsum(0)
    on_card, out = offsets.int().cuda(), torch.full((P + 1, N), 7.0, dtype=torch.bfloat16, device="cuda")
    a = _C.MoeGemmArgs()
    a.x, a.weights, a.out, a.expert_offsets = x.data_ptr(), w.data_ptr(), out.data_ptr(), on_card.data_ptr()
    a.a_rows_div, a.max_rows, a.K, a.N, a.x_stride_m, a.out_stride_m, a.w_stride_e = 1, P, K, N, K, N, N * K
    a.local_expert_begin, a.local_expert_end = local
    assert lib.hymeta_moe_gemm_rank(C.byref(a), total, NONE, 0.0, 0.0, torch.cuda.current_stream().cuda_stream) == 0
    for e in range(E):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        want = (x[lo:hi].float() @ w[e].float().t()).bfloat16() if local[0] <= e < local[1] else torch.full_like(out[lo:hi], 7.0)
        assert torch.equal(out[lo:hi], want), f"expert {e}"
    assert bool((out[P] == 7.0).all())


def test_what_the_tiles_do_not_take():
    """No activation for a problem of few rows; int8 knows the quantised path's silu only."""
    from vllm_hymeta import _C
    lib = _C.load()
    x = torch.zeros(4096, 512, dtype=torch.int8, device="cuda")
    w = torch.zeros(4, 5120, 512, dtype=torch.int8, device="cuda")
    scale = torch.ones(4 * 5120, device="cuda")
    out = torch.zeros(4096, 2560, dtype=torch.bfloat16, device="cuda")
    offsets = torch.tensor([0, 4, 8, 12, 16], dtype=torch.int32, device="cuda")
    ptr = lambda t: C.c_void_p(t.data_ptr())      # noqa: E731
    a = _C.MoeGemmArgs()
    a.x, a.weights, a.out, a.expert_offsets = ptr(x), ptr(w), ptr(out), ptr(offsets)
    a.max_rows, a.K, a.N, a.local_expert_end = 16, 512, 5120, 4
    a.x_stride_m, a.out_stride_m, a.w_stride_e = 512, 2560, 5120 * 512
    a.operand_dtype, a.x_scale, a.w_scale = _C.HYMETA_I8, ptr(scale), ptr(scale)
    unsupported = -2
    assert lib.hymeta_moe_gemm_activates(C.byref(a)) == 0
    assert lib.hymeta_moe_gemm_act(C.byref(a), SILU, 0.0, 0.0, None) == unsupported
    a.max_rows = 4096
    assert lib.hymeta_moe_gemm_activates(C.byref(a)) == 1
    assert lib.hymeta_moe_gemm_act(C.byref(a), CLAMPED, 7.0, 1.702, None) == unsupported
    assert lib.hymeta_moe_gemm_act(C.byref(a), 4, 0.0, 0.0, None) == -1


@pytest.mark.parametrize("M,N,K", [(1030, 32768, 256), (2307, 14336, 320)])      # ragged last row tiles; whole rounds and halves behind them
def test_gate_up_of_a_prompt(M, N, K):
    """The activation in the epilogue: the bits of the exact sums, rounded, then the activation's own launch."""
    from vllm_hymeta import hip_ops
    g = gen(5)
    x = _ints(g, -3, 3, M, K).to(torch.bfloat16).cuda()
    w = _ints(g, -2, 2, N, K).to(torch.bfloat16).cuda()
    assert hip_ops.gemm_silu_mul_supported(x, w)
    out = hip_ops.gemm_silu_mul(x, w)
    assert torch.equal(out, hip_ops.silu_and_mul((x.float() @ w.float().t()).to(torch.bfloat16)))
    # a view of wider rows; a shape of too few tiles is left to the library
    wide = torch.zeros(M, K + 64, dtype=torch.bfloat16, device="cuda")
    wide[:, :K] = x
    assert torch.equal(hip_ops.gemm_silu_mul(wide[:, :K], w), out)
    assert not hip_ops.gemm_silu_mul_supported(x[:300], w[:8192])


@pytest.mark.parametrize("M", [300, 1030, 5000])      # too few tiles, a prompt in tiles, too many
def test_gated_block_of_a_prompt(M):
    """The side families' gated block has one activation for prompts of any length: silu_mul of the rounded exact sums (in
    sixteenths, up to +-24: an exponential formed less exactly gives other bits in some of them)."""
    from vllm_hymeta import hip_ops
    from vllm_hymeta.linear import HymetaLinear
    from vllm_hymeta.models.feed_forward import SiluGluMLP
    g = gen(13)
    K, N = 256, 32768
    x, w = (_ints(g, -3, 3, M, K) / 16).bfloat16().cuda(), _ints(g, -3, 3, N, K).bfloat16().cuda()
    assert hip_ops.gemm_silu_mul_supported(x, w) == (M == 1030)
    h = (x.float() @ w.float().t()).bfloat16()
    want, fast = hip_ops.silu_mul(h), hip_ops.silu_and_mul(h)
    assert not torch.equal(want, fast)
    down = HymetaLinear.from_weight(torch.eye(256, N // 2, dtype=torch.bfloat16, device="cuda"))      # the first 256 columns
    out = SiluGluMLP(HymetaLinear.from_weight(w), down)(x)
    assert torch.equal(out, want[:, :256])
    if M == 1030:
        assert torch.equal(hip_ops.gemm_silu_mul(x, w, exact=True), want) and torch.equal(hip_ops.gemm_silu_mul(x, w), fast)


@pytest.mark.parametrize("M,N,K", [
    (1030, 4608, 512), (300, 16384, 640), (5000, 1024, 1024),
    (1024, 4096, 512), (1025, 4096, 512),        # a tile of 128 x 128 for every unit, and more
    (640, 11264, 512), (1025, 11264, 512),       # more large tiles than are cut in halves, small ones for every place, and more
    (400, 8192, 3072), (300, 9472, 3072),        # a longer K, few rows
    (600, 8192, 3072),                           # halves with an activation
    (8493, 1024, 512), (16641, 1024, 512),       # row tiles of two and of three sweeps over the columns
    (1025, 4096, 2048), (520, 14336, 3072),      # a K that pays for the large tiles
    (300, 50944, 512), (500, 50944, 512),        # half-empty large tiles, and nearly filled ones
    (150, 50944, 512), (256, 49152, 640),        # one row tile: eight waves
    (200, 12544, 3072), (130, 49280, 512),       # ... too few of them, and columns that are no whole tiles
])
@pytest.mark.parametrize("gated", [False, True])
def test_w8a8_linear_of_a_prompt(M, N, K, gated):
    """Exact int32 sums, (sum * x_scale) * w_scale + bias in one fused step, one rounding: powers of two keep all of it exact
    but the bias's sum, which fp64 gives to the same bf16 (24 + 8 bits)."""
    from vllm_hymeta import hip_ops
    g = gen(6)
    xq = _ints(g, -127, 127, M, K).to(torch.int8)
    xq[:, 0] = 127                                                   # the row's largest: its scale is exactly the one chosen
    scale = 2.0 ** _ints(g, -9, -5, M).float()
    x = (xq.float() * scale[:, None]).to(torch.bfloat16).cuda()      # 7 bits: exact
    w = _ints(g, -127, 127, N, K).to(torch.int8).cuda()
    ws = (2.0 ** _ints(g, -9, -6, N).float()).cuda()
    bias = _ints(g, -64, 64, N).to(torch.bfloat16).cuda()
    q, s = hip_ops.w8a8_quantize(x)
    assert torch.equal(q.cpu(), xq) and torch.equal(s.cpu(), scale)
    sums = (q.double() @ w.double().t()) * s.double()[:, None] * ws.double()
    if gated:
        out = hip_ops.gemm_silu_mul(x, w, ws)
        ref = hip_ops.silu_and_mul(sums.to(torch.bfloat16))
    else:
        out = hip_ops.w8a8_gemm(x, w, ws, bias=bias)
        ref = (sums + bias.double()).float().to(torch.bfloat16)
    assert torch.equal(out, ref)


@pytest.mark.parametrize("M,N,K,slices,bias,pitch", [
    (257, 3584, 18944, 9, False, 18944),      # a last row tile of one row
    (512, 256, 24704, 16, True, 24720),       # the most slices, of 24 and 25 steps; x in rows of a wider tensor
    (1025, 3584, 7232, 3, True, 7232),        # slices of 37 and 38 steps, a die's tiles from two of them
    (2048, 1024, 12352, 8, False, 12352),
    (2048, 3584, 14336, 2, False, 14336),     # two slices: K of four times the weight rows
])
def test_a_product_cut_along_k(M, N, K, slices, bias, pitch):
    from vllm_hymeta import hip_ops
    from vllm_hymeta.linear import HymetaLinear
    g = gen(11)
    x, w = _ints(g, -3, 3, M, pitch).bfloat16().cuda()[:, :K], _ints(g, -2, 2, N, K).bfloat16().cuda()
    b = _ints(g, -9, 9, N).bfloat16().cuda() if bias else None
    sums = hip_ops.bf16_gemm_sliced(x, w, b)
    assert sums.desc.splits == slices
    ref = x.float() @ w.float().t()           # sums below 2^24: exact in any order
    want = (ref if b is None else ref + b.float()).bfloat16()
    assert torch.equal(sums.tensor(), want)
    layer = HymetaLinear.from_weight(w, b)
    assert torch.equal(layer(x), want)
    residual, weight = torch.zeros(M, N, dtype=torch.bfloat16, device="cuda"), torch.ones(N, dtype=torch.bfloat16, device="cuda")
    deferred = layer(x, defer=True)
    assert isinstance(deferred, hip_ops.PartialSums)
    hip_ops.add_rmsnorm(deferred, weight, residual=residual)
    assert torch.equal(residual, want)


@pytest.mark.parametrize("M,N,K,deferred,reduced", [
    (3072, 1024, 8192, False, False), (1536, 2048, 8192, False, False), (900, 3072, 8192, False, False),      # not deep
    (2561, 1536, 8960, False, False), (2560, 1536, 8960, True, True),             # rows that leave units idle, of a narrow matrix
    (1025, 3584, 9472, True, False), (1024, 3584, 9472, True, True),              # ... and of a wider one, where a launch reduces them
    (1025, 3584, 18944, True, True),                                              # deep enough
    (3072, 2048, 16384, False, False), (1500, 4096, 16384, False, False),         # two slices of too few tiles or columns
    (330, 8192, 16384, False, False), (330, 8192, 16448, True, True),             # rows whole 32 KB apart
    (2048, 1024, 16384, True, True),                                              # few tiles
])
def test_products_that_the_library_has_sooner(M, N, K, deferred, reduced):
    from vllm_hymeta import hip_ops
    from vllm_hymeta.linear import HymetaLinear
    x, w = torch.ones(M, K, dtype=torch.bfloat16, device="cuda"), torch.ones(N, K, dtype=torch.bfloat16, device="cuda")
    assert (hip_ops.bf16_gemm_sliced(x, w) is not None) == deferred
    assert (hip_ops.bf16_gemm_sliced(x, w, reduced=True) is not None) == reduced
    layer = HymetaLinear.from_weight(w)
    assert isinstance(layer(x, defer=True), hip_ops.PartialSums) == deferred
    assert bool((layer(x) == K).all()) or K % 256 != 0                             # (exact in bf16 where K is)


def test_the_slices_memory():
    """Two prompts' partial sums beside each other, on their own stream and on another one; given back afterwards."""
    from vllm_hymeta import hip_ops
    M, N, K = 512, 3584, 18944
    g = gen(19)
    x, w = _ints(g, -3, 3, M, K).bfloat16().cuda(), _ints(g, -2, 2, N, K).bfloat16().cuda()
    want = (x.float() @ w.float().t()).bfloat16()
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    one, two = hip_ops.bf16_gemm_sliced(x, w), hip_ops.bf16_gemm_sliced(-x, w)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        first = one.tensor()
        del one
    hip_ops.bf16_gemm_sliced(2 * x, w)                     # (does not land in memory that the other stream still reads)
    torch.cuda.current_stream().wait_stream(side)
    second = two.tensor()
    assert torch.equal(first, want) and torch.equal(second, -want)
    torch.cuda.synchronize()
    del first, second, two, side
    again = hip_ops.bf16_gemm_sliced(x, w).tensor()        # (the allocator looks for blocks that other streams are done with)
    assert torch.equal(again, want)
    del again
    assert torch.cuda.memory_allocated() == before
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = hip_ops.bf16_gemm_sliced(x, w).tensor()
    for sign in (1, -1, 1):
        x.mul_(sign)
        graph.replay()
        assert torch.equal(out, hip_ops.bf16_gemm_sliced(x, w).tensor())


def test_a_linear_that_is_more_than_its_kernel():
    """What torch's linear does beside the product stays: a bias that is broadcast or does not fit, gradients of either direction,
    autocast's type.  (Sums of small integers: exact.)"""
    from vllm_hymeta import hip_ops
    from vllm_hymeta.linear import HymetaLinear
    M, N, K = 300, 3584, 18944
    g = gen(17)
    x, w = _ints(g, -3, 3, M, K).bfloat16().cuda(), _ints(g, -2, 2, N, K).bfloat16().cuda()
    ref = x.float() @ w.float().t()
    assert hip_ops.bf16_gemm_sliced(x, w) is not None
    one = torch.full((1,), 5.0, dtype=torch.bfloat16, device="cuda")
    assert torch.equal(HymetaLinear.from_weight(w, one)(x), (ref + 5).bfloat16())
    with pytest.raises(RuntimeError):
        HymetaLinear.from_weight(w, torch.zeros(N - 1, dtype=torch.bfloat16, device="cuda"))(x)
    bias = torch.zeros(N, dtype=torch.bfloat16, device="cuda", requires_grad=True)
    HymetaLinear.from_weight(w, bias)(x).sum().backward()
    assert torch.equal(bias.grad, torch.full_like(bias, M))
    layer, ad = HymetaLinear.from_weight(w), torch.autograd.forward_ad
    with torch.no_grad(), ad.dual_level():
        y = ad.unpack_dual(layer(ad.make_dual(x, 2 * x)))
    assert torch.equal(y.primal, ref.bfloat16()) and torch.equal(y.tangent, (2 * ref).bfloat16())
    with torch.no_grad(), torch.autocast("cuda", torch.float16):
        assert layer(x).dtype == torch.float16


@pytest.mark.parametrize("M,N,K", [(256, 3584, 18944), (300, 3584, 3584), (2048, 3584, 9472), (300, 3520, 18944), (300, 3584, 18976), (4096, 3584, 18944)])
def test_products_that_are_not_cut(M, N, K):
    from vllm_hymeta import hip_ops
    x, w = torch.ones(M, K, dtype=torch.bfloat16, device="cuda"), torch.zeros(N, K, dtype=torch.bfloat16, device="cuda")
    assert hip_ops.bf16_gemm_sliced(x, w) is None
    if M > 256 and K % 64 == 0:
        assert hip_ops.bf16_gemm_sliced(x[:, : K - 64], w[:, : K - 64]) is None      # weight rows that are not next to each other
