"""Which prompts' portions linear attention in chunks cuts into segments (``scan_segments`` in csrc/chunk_scan.h), and that the
workspace's bound holds for every cut, by the very code on the host."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "chunk_scan.h"
using namespace hymeta;

// pieces of a portion of `rows` rows, of `portions` of them beside `singles` single ones (1: not cut)
static int pieces(int portions, int rows, int singles, int heads, int v_dim, bool silu) {
  const ScanSegments sg = scan_segments(portions * rows + singles, portions + singles, heads, v_dim, rows, silu);
  return sg.count == 0 ? 1 : (rows + sg.rows - 1) / sg.rows;
}

int main(int argc, char** argv) {
  if (argc == 7) {
    int v[6];
    for (int i = 0; i < 6; ++i) v[i] = std::atoi(argv[i + 1]);
    std::printf("%d\n", pieces(v[0], v[1], v[2], v[3], v[4], v[5] != 0));
    return 0;
  }
  // random steps: a cut portion has at least three pieces of whole chunks, and the numbers that its step needs fit the workspace
  // that is asked for with as many sequences and as long a portion, or more
  uint64_t seed = 1;
  auto below = [&](uint64_t n) { return static_cast<int>((seed = seed * 6364136223846793005ull + 1442695040888963407ull, seed >> 33) % n); };
  auto size = [&](int bits) { return 1 + below(1ull << below(bits + 1)); };
  const int widths[] = {32, 64, 96, 128, 256, 512};
  long cut = 0;
  for (int i = 0; i < 3000000; ++i) {
    const int heads = size(6), v_dim = widths[below(6)], most = size(15), seqs = size(9), D = 64;
    const int tokens = seqs + below(static_cast<uint64_t>(seqs) * most - seqs + 1);
    const ScanSegments sg = scan_segments(tokens, seqs, heads, v_dim, most, below(2) != 0);
    if (sg.count == 0) continue;
    ++cut;
    const size_t room = scan_workspace_bytes(seqs + (below(2) ? 0 : size(6)), heads, D, v_dim, most + (below(2) ? 0 : size(8)));
    if (sg.rows % kScanRows != 0 || (most + sg.rows - 1) / sg.rows < 3 || scan_segment_bytes(sg.count, heads, D, v_dim) > room) {
      std::printf("tokens %d sequences %d heads %d columns %d longest %d: %d of %d rows, room %zu\n", tokens, seqs, heads, v_dim, most, sg.count, sg.rows, room);
      return 1;
    }
  }
  std::printf("%ld\n", cut);
  return cut > 100000 ? 0 : 1;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    at = tmp_path_factory.mktemp("segments")
    (at / "segments.hip").write_text(PROGRAM)
    subprocess.run([HIPCC, "-O1", "-std=c++17", "--offload-host-only", "-w", "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "vllm-hymeta_amd", "csrc"),
                    str(at / "segments.hip"), "-o", str(at / "segments")], check=True, capture_output=True)
    return str(at / "segments")


def test_every_cut_has_three_pieces_and_fits_the_workspace(program):
    assert subprocess.run([program], capture_output=True, text=True, timeout=300).returncode == 0


@pytest.mark.parametrize("portions,rows,singles,heads,columns,silu,pieces", [
    (1, 191, 0, 16, 128, 1, 1), (1, 192, 0, 16, 128, 1, 3), (1, 192, 0, 16, 128, 0, 1), (1, 200, 0, 16, 128, 1, 1), (3, 200, 0, 28, 128, 0, 1),      # two pieces after rounding
    (1, 256, 0, 16, 128, 0, 4), (1, 256, 0, 28, 128, 0, 1), (1, 256, 0, 28, 128, 1, 4), (2, 256, 0, 28, 128, 1, 1),        # what they save against what they cost
    (1, 300, 0, 28, 128, 0, 3), (2, 300, 0, 28, 128, 0, 1), (2, 300, 0, 16, 128, 0, 3), (3, 500, 0, 28, 128, 0, 3),
    (1, 256, 0, 56, 64, 0, 4), (2, 256, 0, 56, 64, 0, 1), (3, 400, 0, 56, 64, 0, 1), (3, 260, 0, 32, 64, 0, 3), (5, 450, 0, 28, 64, 0, 1),
    (1, 8192, 0, 28, 128, 1, 9), (1, 2048, 0, 16, 128, 0, 16), (1, 2048, 31, 16, 128, 0, 8), (1, 2048, 63, 7, 128, 0, 32),      # more than ten, beside short portions
    (1, 2048, 0, 16, 64, 0, 32), (1, 2048, 63, 16, 64, 0, 8), (1, 2048, 63, 16, 64, 1, 32), (1, 2048, 100, 16, 64, 1, 8),
    (1, 2048, 0, 32, 64, 0, 8), (1, 2048, 0, 28, 64, 0, 16), (1, 1000, 255, 28, 128, 0, 4), (1, 575, 255, 28, 128, 0, 1),
])
def test_which_portions_are_cut(program, portions, rows, singles, heads, columns, silu, pieces):
    out = subprocess.run([program, *map(str, (portions, rows, singles, heads, columns, silu))], capture_output=True, text=True, check=True, timeout=60)
    assert int(out.stdout) == pieces
