"""The tiled products' matrix instructions are inline assembly, whose results the compiler does not know to be late: no
accumulator may be moved between the instructions of a run and the wait that ends it."""
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
    flags = ["-O3", "-std=c++17", "--offload-arch=gfx950", "-I", os.path.join(PKG, "..", "include"), "-I", os.path.join(PKG, "csrc"),
             "-ffp-contract=fast", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
    subprocess.run([HIPCC, *flags, "-S", "--cuda-device-only", os.path.join(PKG, "csrc", "tile_gemm.hip"), "-o", str(out)],
                   check=True, capture_output=True)
    text = out.read_text()
    kernels = re.split(r"\n(?=_ZN6hymeta\S*tile_gemm_kernel\S*:)", text)[1:]
    assert len(kernels) >= 6
    for body in kernels:
        body = body.split("s_endpgm")[0] if body.count("s_endpgm") == 1 else body
        runs = 0
        for block in re.split(r"\n(?=\.LBB\d+_\d+:)", body):
            in_flight = False
            for line in block.splitlines():
                line = line.split(";")[0]
                if "v_mfma" in line:
                    assert re.search(r"v_mfma\S+ (a\[\d+:\d+\]), v\[\S+\], v\[\S+\], \1", line), line      # in place
                    in_flight, runs = True, runs + 1
                elif "s_nop 9" in line:
                    in_flight = False
                elif in_flight:
                    assert not re.search(r"\ba\d|\ba\[", line), line
            # a run that goes on in the next block: its first instruction is another product or the wait, by the order that
            # the source fixes; a block that ends in flight must not hold anything else
        assert runs >= 192
        assert not re.search(r"scratch_(load|store)", body), "a spill would wait for every copy in flight"
