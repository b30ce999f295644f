"""Which columns and rows the positive-definite correction's visit test reads
(cm1_amd/csrc/cm1g_pdef_visit.h), compiled for the CPU: for every domain width
and every tile, both neighbours of every cell of the tile, wrapped (periodic)
or clamped (open) at the domain's ends, are in the tile's own 64-column word
or among the side columns read; and the same for rows."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include "cm1g_pdef_visit.h"

static int nb(int m, int n, bool per) { return m < 1 ? (per ? n : 1) : m > n ? (per ? 1 : n) : m; }

int main() {
  long seen = 0, missed = 0, outside = 0;
  for (int n = 8; n <= 700; n++)
    for (int per = 0; per < 2; per++) {
      for (int t = 0; 64 * t < n; t++) {
        const int i0 = 1 + 64 * t;
        const int l = pdef_side_col(i0, n, false, per), r = pdef_side_col(i0, n, true, per);
        outside += l < 1 || l > n || r < 1 || r > n;
        for (int i = i0; i < i0 + 64 && i <= n; i++)
          for (int d = -1; d <= 1; d += 2) {
            const int m = nb(i + d, n, per);
            seen++;
            if ((m - 1) / 64 != t && m != l && m != r) {
              if (!missed) std::printf("n %d periodic %d cell %d neighbour %d\n", n, per, i, m);
              missed++;
            }
          }
      }
      for (int j0 = 1; j0 <= n; j0 += 4)
        for (int j = j0; j < j0 + 4 && j <= n; j++)
          for (int d = -1; d <= 1; d++) {
            const int m = nb(j + d, n, per);
            bool found = false;
            for (int q = 0; q < 6; q++) {
              const int row = pdef_wrap(j0 - 1 + q, n, per);
              outside += row < 1 || row > n;
              found = found || row == m;
            }
            seen++;
            missed += !found;
          }
    }
  std::printf("%ld %ld %ld\n", seen, missed, outside);
}
"""


def test_visit_reads_every_neighbour(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    src, exe = tmp_path / "visit.cpp", str(tmp_path / "visit")
    src.write_text(SRC)
    subprocess.run([cxx, "-O2", "-I", os.path.join(ROOT, "cm1_amd", "csrc"), str(src), "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    seen, missed, outside = (int(v) for v in out.split()[-3:])
    assert seen > 1_000_000 and missed == 0 and outside == 0, out
