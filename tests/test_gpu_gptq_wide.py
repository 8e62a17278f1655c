"""4-bit GPTQ products of 33 to 128 rows whose 128-column tiles leave a remainder behind whole rounds of compute units: tiles of 160
columns, the last one ragged by every remainder, groups of 32 / 64 / 128, one and two blocks of 64 rows.

Bound: the outputs are bf16 (2^-9 of each value at most); sums of 512 products x (128 + q) less (128 + z) times the sum of x, in fp32,
lose below 2^-24 sqrt(512) 2^5 of the result's norm (128 + q is at most 2^5 times q's spread); together below 2^-9 + 2^-14."""
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
    worst = (out.double() - ref).norm(dim=0) / ref.norm(dim=0)             # (2^-9 of each value: a column's norm too)
    assert float(worst.max()) < 2 ** -8 and float((out.double() - ref).norm()) < (2 ** -9 + 2 ** -14) * float(ref.norm())
    assert bool((behind[M:] == 7).all()) and bool((behind[:, N:] == 7).all())
