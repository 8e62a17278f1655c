"""4-bit GPTQ products of up to 16 and of 33 to 128 rows whose tiles leave a remainder behind whole rounds of compute units: tiles of
80 and 160 columns, the last one ragged by every remainder, groups of 32 / 64 / 128, one and two blocks of 64 rows.

Bound: the outputs are bf16 (2^-8 of each value at most, over many values 2^-8 / sqrt(3) of their norm times the 0.74 that a uniform
mantissa leaves: below 2^-9); sums of up to 1152 products x (128 + q) less (128 + z) times the sum of x, in fp32,
lose below 2^-24 sqrt(1152) 2^5 of the result's norm (128 + q is at most 2^5 times q's spread); together below 2^-9 + 2^-14."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K,G,M,half,bias", [
    (37888, 512, 128, 64, True, False),       # 128 of the last tile's 160 columns
    (32896, 1024, 64, 33, False, True),       # 96
    (33024, 512, 32, 50, True, True),         # 64
    (33152, 256, 128, 64, False, False),      # 32
    (40960, 768, 64, 63, True, True),         # all, a tile for every compute unit
    (18944, 512, 128, 65, True, True),        # a second block of one row
    (37888, 512, 128, 128, False, True),      # two rounds
    (32768, 512, 128, 64, True, True),        # whole rounds of 128 columns
    (41088, 512, 128, 64, True, False),       # one tile of 160 too many: 128 columns and slices
    (57344, 512, 64, 65, True, True),         # three rounds of 160 in place of three and a half: 128 columns and slices
    # up to 16 rows, tiles of 80: the last one with 48, 64, 32, 16 and all of its columns
    (37888, 512, 128, 1, True, True),
    (33024, 1152, 64, 16, False, False),      # an odd number of groups a wave
    (32832, 256, 32, 5, True, True),
    (32896, 640, 128, 16, False, True),
    (40960, 512, 64, 9, True, False),
    (41024, 512, 128, 16, True, True),        # one too many: tiles of 64
    (18944, 512, 128, 16, False, True),       # one of 80 in place of two: tiles of 64
])
def test_columns_of_every_tile(N, K, G, M, half, bias):
    from vllm_hymeta import hip_ops
    g = torch.Generator(device="cuda").manual_seed(N + M)
    f = dict(device="cuda", generator=g)
    q, z = torch.randint(0, 16, (K, N), **f), torch.randint(0, 16, (K // G, N), **f)
    s = (0.005 + 0.02 * torch.rand(K // G, N, **f)).to(torch.float16 if half else torch.bfloat16)
    qw = sum(q.view(K // 8, 8, N)[:, j] << (4 * j) for j in range(8))
    zw = sum(z.view(K // G, N // 8, 8)[:, :, j] << (4 * j) for j in range(8))
    i32 = lambda t: torch.where(t >= 1 << 31, t - (1 << 32), t).int()      # noqa: E731
    x = torch.randn(M, K, **f).bfloat16()
    b = torch.randn(N, **f).bfloat16() if bias else None
    behind = torch.full((M + 1, N + 64), 7.0, dtype=torch.bfloat16, device="cuda")
    out = hip_ops.gptq_gemm(x, i32(qw), i32(zw), s, 4, G, bias=b, out=behind[:M, :N])
    w = ((q.double().view(K // G, G, N) - (z.double() + 1)[:, None]) * s.double()[:, None]).view(K, N)
    ref = x.double() @ w + (0 if b is None else b.double())
    # each value: its rounding (8 significant bits: half a unit in the last place is 2^-8 of it at most), and of at most G + K / G + 8 additions of terms below 143 s |x| each 2^-24 of what is summed
    lost = 2 ** -24 * (G + K // G + 8) * 143 * float(s.max()) * x.double().abs().sum(1, keepdim=True)
    assert bool(((out.double() - ref).abs() <= 2 ** -8 * ref.abs() * 1.01 + lost).all())
    assert float((out.double() - ref).norm()) < (2 ** -9 + 2 ** -14) * float(ref.norm())
    assert bool((behind[M:] == 7).all()) and bool((behind[:, N:] == 7).all())
