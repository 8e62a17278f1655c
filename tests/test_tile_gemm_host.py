"""The tiled products' matrix instructions are inline assembly, whose results the compiler does not know to be late: no
accumulator may be moved between the instructions of a run and the wait that ends it."""
import ctypes as C
import os
import re
import shutil
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-hymeta_amd")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_nothing_touches_an_accumulator_in_flight(tmp_path):
    out = tmp_path / "tile_gemm.s"
    # the very command that the library is built with, to assembly in place of an object
    dry = subprocess.run(["make", "-C", PKG, "-n", "-B", os.path.join(PKG, "build", "tile_gemm.o")], check=True, capture_output=True, text=True).stdout
    command = next(line.split() for line in dry.splitlines() if "tile_gemm.hip" in line and "-o" in line.split())
    at = command.index("-o")
    command = [HIPCC, *(word for word in command[1:at] + command[at + 2:] if word not in ("-c", "-MMD", "-MP")), "-S", "--cuda-device-only", "-o", str(out)]
    assert "-packed-fp32-ops" in command and "--offload-arch=gfx950" in command
    subprocess.run(command, check=True, capture_output=True, cwd=PKG)
    text = out.read_text()
    kernels = re.split(r"\n(?=_ZN6hymeta\S*tile_gemm_kernel\S*:)", text)[1:]
    assert len(kernels) >= 6
    for body in kernels:
        body = body.split("s_endpgm")[0] if body.count("s_endpgm") == 1 else body
        runs, in_flight = 0, False                   # (over labels too: a copy's branch stands inside a run of products)
        for line in body.splitlines():
            line = line.split(";")[0]
            if "v_mfma" in line:
                assert re.search(r"v_mfma\S+ (a\[\d+:\d+\]), v\[\S+\], v\[\S+\], \1", line), line      # in place
                in_flight, runs = True, runs + 1
            elif "s_nop 9" in line:
                in_flight = False
            elif in_flight:
                assert not re.search(r"\ba\d|\ba\[", line), line
        assert runs >= 192
        assert not re.search(r"scratch_(load|store)", body), "a spill would wait for every copy in flight"


def test_rows_of_x_that_run_backwards():
    """Their offsets are unsigned in the tiles: grouped products leave such rows to the kernel with 64-bit addresses, products of one
    matrix refuse them (before anything is launched)."""
    from vllm_hymeta import _C
    lib, unsupported = _C.load(), -2
    a = _C.MoeGemmArgs()
    a.max_rows, a.K, a.N, a.local_expert_end, a.x_stride_m, a.out_stride_m, a.w_stride_e = 4096, 512, 5120, 4, 512, 2560, 5120 * 512
    assert lib.hymeta_moe_gemm_activates(C.byref(a)) == 1
    a.x_stride_m = -512
    assert lib.hymeta_moe_gemm_activates(C.byref(a)) == 0
    b, partials = _C.Bf16GemmArgs(), _C.GemmPartials()
    b.x = b.weight = b.out = b.workspace = 1 << 20
    b.workspace_bytes, b.M, b.K, b.N, b.x_stride_m, b.w_stride_n, b.out_stride_m = 64 << 20, 512, 18944, 3584, -18944, 18944, 3584
    assert lib.hymeta_bf16_gemm_sliced(C.byref(b), C.byref(partials), None) == unsupported
    b.M, b.K, b.N, b.x_stride_m, b.w_stride_n, b.out_stride_m = 1280, 3584, 37888, -3584, 3584, 18944
    assert lib.hymeta_bf16_gemm_takes(1280, 3584, 37888, 1) == 1
    assert lib.hymeta_bf16_gemm_silu_mul(C.byref(b), None) == unsupported


def test_rows_that_a_ranks_experts_can_expect():
    """8 experts of 14336 x 8192 and 1200 pairs: 150 rows each fill the tiles, 75 each, where 16 share the pairs, do not; from 192 pairs an
    expert the tiles are used either way, and experts that nearly fill one tile go without the activation."""
    from vllm_hymeta import _C
    lib = _C.load()
    a = _C.MoeGemmArgs()
    a.K, a.N, a.local_expert_end, a.x_stride_m, a.out_stride_m, a.w_stride_e = 8192, 14336, 8, 8192, 7168, 14336 * 8192
    for pairs, own, of16 in ((1100, 0, 0), (1200, 1, 0), (1535, 0, 0), (1536, 0, 1), (1919, 0, 1), (1920, 1, 1), (3000, 1, 0), (4000, 1, 1)):
        a.max_rows = pairs
        assert (lib.hymeta_moe_gemm_activates(C.byref(a)), lib.hymeta_moe_gemm_rank_activates(C.byref(a), 16)) == (own, of16), pairs
        assert lib.hymeta_moe_gemm_rank_activates(C.byref(a), 8) == own, pairs


@pytest.mark.parametrize("M,K,N,takes", [
    (896, 3584, 37888, 1), (2048, 3584, 37888, 1), (3328, 3584, 37888, 1), (700, 3584, 37888, 0), (4097, 3584, 37888, 0),      # 513 to 2048 tiles
    (1030, 256, 32768, 1), (2307, 320, 14336, 1), (8192, 960, 6144, 1),      # a short K
    (2048, 8192, 57344, 0), (1280, 5120, 27648, 0),                          # a long one
    (800, 1600, 35072, 0), (1024, 1600, 35072, 1),                           # rows that leave a fifth of the rounds empty
    (5000, 3584, 7168, 0),                                                   # few columns
    (3328, 3584, 10496, 0), (2816, 3584, 19200, 1), (3000, 2048, 12800, 1), (4451, 2048, 9216, 0),
    (1024, 2816, 36864, 0), (1024, 2816, 37120, 1),                          # a multiple of 2048 columns, and none
    (4474, 4032, 9984, 0), (2560, 3840, 18944, 0), (2560, 3584, 18944, 1),   # a long K
    (2231, 3584, 18944, 0), (1900, 3584, 37888, 1),                          # a last round of half to three quarters of the units, of three and of five
    (1152, 3584, 52480, 0), (769, 3584, 37888, 1), (1694, 2048, 28672, 0),   # rounds filled to 78 %; to 67 % where they are few; to 80 %
    (769, 2560, 37888, 1), (1600, 3584, 19200, 0), (769, 2048, 37888, 0),    # ... few with few tiles in the last one; a short K
])
def test_gate_up_projections_that_run_in_tiles(M, K, N, takes):
    from vllm_hymeta import _C
    assert _C.load().hymeta_bf16_gemm_takes(M, K, N, 1) == takes


@pytest.mark.parametrize("experts,total,K,N,int8,pairs,takes", [
    # from nine rows an expert on, but not columns or a K that no tile takes
    (16, 16, 3584, 9472, 0, 128, 0), (16, 16, 3584, 9472, 0, 129, 1), (16, 16, 3584, 9472, 1, 128, 0), (16, 16, 3584, 9472, 1, 129, 1),
    (16, 16, 3584, 9536, 0, 600, 0), (16, 16, 3616, 9472, 0, 600, 0), (16, 16, 3616, 9472, 1, 600, 0),
    # experts that nearly fill one tile go without from a K of 5120 on, from 176 rows (448 tiles: three quarters of their last round of the chip)
    (8, 8, 8192, 14336, 0, 1407, 1), (8, 8, 8192, 14336, 0, 1408, 0), (8, 8, 8192, 14336, 0, 1919, 0), (8, 8, 8192, 14336, 0, 1920, 1),
    (8, 8, 5056, 14336, 0, 1600, 1), (8, 8, 5120, 14336, 0, 1600, 0), (8, 8, 8192, 14336, 1, 1600, 1),
    # ... those that a rank's experts can expect
    (8, 16, 8192, 14336, 0, 2815, 1), (8, 16, 8192, 14336, 0, 2816, 0), (8, 16, 8192, 14336, 0, 3840, 1),
    # from 160 where the tiles fill the chip once, or their last round (256 and 512 tiles); never below 148 of them (120), or with 64 and
    # fewer in the second round (288, 320, and 324)
    (8, 8, 8192, 8192, 0, 1279, 1), (8, 8, 8192, 8192, 0, 1280, 0), (16, 16, 8192, 8192, 0, 2559, 1), (16, 16, 8192, 8192, 0, 2560, 0),
    (4, 4, 8192, 7680, 0, 700, 1), (4, 4, 8192, 7680, 0, 900, 1), (8, 8, 8192, 9216, 0, 1900, 1), (8, 8, 8192, 10240, 0, 1900, 1),
    (12, 12, 8192, 6912, 0, 2111, 1), (12, 12, 8192, 6912, 0, 2112, 0),
])
def test_products_with_the_activation_in_the_epilogue(experts, total, K, N, int8, pairs, takes):
    """Which grouped products have their activation inside (``hymeta_moe_gemm_glu``), on either side of every limit."""
    from vllm_hymeta import _C
    a = _C.MoeGemmArgs()
    a.max_rows, a.K, a.N, a.local_expert_end, a.x_stride_m, a.out_stride_m, a.w_stride_e = pairs, K << int8, N, experts, K << int8, N // 2, (K << int8) * N
    a.operand_dtype = _C.HYMETA_I8 if int8 else _C.HYMETA_BF16
    assert _C.load().hymeta_moe_gemm_glu_takes(C.byref(a), total) == takes
