"""The bytes that the tiled GEMM's last, half-filled K stage reads (csrc/gemm_stage.h), checked on the CPU.

The 256-row tiles load K in stages of 128 bytes; when K is an odd multiple of 64 bytes the last stage is half
a stage.  An operand may be a column range of a wider matrix (row stride > K), whose last row ends with the
allocation, so no lane may read past byte K of its row: the program below compiles the kernel's own offset
arithmetic with the host compiler, walks every wave, load and lane of a tile at the matrix's ragged end, and
requires each load to lie inside its row or to be refused by the buffer's range check (an offset of at least
rows x stride), with every chunk of the half stage loaded once per row.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "minicpm5-vllm-tpu_amd", "csrc")

SRC = r"""
#include "gemm_stage.h"
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>
// argv: rows, tile rows, row stride (bytes), K (bytes): the last tile of one operand, eight waves
int main(int, char** v) {
  const uint32_t rows = atoi(v[1]), bm = atoi(v[2]), ld = atoi(v[3]), kb = atoi(v[4]);
  constexpr int BKB = 128, CPR = BKB / 16, RPB = 1024 / BKB, NW = 8;
  const uint32_t m0 = (rows - 1) / bm * bm, at = kb / BKB * BKB;   // the half stage's first K byte
  std::vector<int> seen(bm * CPR);
  for (int w = 0; w < NW; ++w)
    for (uint32_t j = 0; j < bm / RPB / NW; ++j)
      for (int lane = 0; lane < 64; ++lane) {
        const int r = RPB * (w + NW * j) + lane / CPR;
        const uint32_t row = std::min(m0 + r, rows - 1);
        const uint32_t voff = row * ld + 16u * mk::stage_chunk<BKB>(lane, r);
        const uint32_t off = mk::half_stage_offset<BKB>(voff, lane, RPB * w + lane / CPR, at);
        if (off >= (uint64_t)rows * ld) continue;                  // refused
        if (off < row * ld || off + 16 > row * ld + kb) return printf("row %u reads byte %u of %u\n", row, off - row * ld, kb), 1;
        ++seen[r * CPR + (off - row * ld - at) / 16];
      }
  for (uint32_t r = 0; r < bm; ++r)
    for (int c = 0; c < CPR; ++c)
      if (seen[r * CPR + c] != (c < CPR / 2)) return printf("row %u chunk %d loaded %d times\n", r, c, seen[r * CPR + c]), 1;
  return 0;
}
"""


@pytest.fixture(scope="module")
def reads(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("stage")
    (d / "reads.cpp").write_text(SRC)
    subprocess.run([cxx, "-std=c++17", "-O1", f"-I{CSRC}", str(d / "reads.cpp"), "-o", str(d / "reads")], check=True)
    return str(d / "reads")


@pytest.mark.parametrize("rows,tile", [(8100, 256), (1, 256), (2560, 320), (1530, 192)])
@pytest.mark.parametrize("kb,pad", [(64, 0), (192, 0), (192, 16), (1600, 64), (1600, 1600), (4160, 112)])
def test_half_stage_reads_stay_in_their_row(reads, rows, tile, kb, pad):
    r = subprocess.run([reads, str(rows), str(tile), str(kb + pad), str(kb)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
