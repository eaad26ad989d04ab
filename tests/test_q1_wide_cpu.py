"""The many-token product's weight offsets, evaluated by the host compiler: every row-block that a workgroup of the
wide kernel asks for lies inside the matrix, also in a last row group that holds fewer than eight of them."""
import os
import subprocess

from conftest import ROOT

SRC = r"""
#include "q1_wide.h"
constexpr bool inside(int64_t nrb) {
  for (int rg = 0; rg < (nrb + dz::kWideRb - 1) / dz::kWideRb; ++rg)
    for (int i = 0; i < dz::kWideRb; ++i) {
      const int64_t first = (int64_t)rg * dz::kWideRb, rb = first + dz::wide_row_block(rg, i, nrb);
      if (rb < first || rb >= nrb || (first + i < nrb && rb != first + i)) return false;
    }
  return true;
}
constexpr bool all() {
  for (int64_t nrb = 1; nrb <= 67; ++nrb)
    if (!inside(nrb)) return false;
  return inside(258) && inside(3880);  // 16480 and 248320 rows
}
static_assert(all(), "a row-block outside the matrix");
"""


def test_row_blocks_inside_the_matrix(tmp_path):
    from daiza_amd import build
    src = tmp_path / "wide.hip"
    src.write_text(SRC)
    r = subprocess.run([build.HIPCC, "--offload-host-only", "-fsyntax-only", "-std=c++17", "-I" + os.path.join(ROOT, "include"),
                        "-I" + build.CSRC, str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
