"""Coefficient columns the device walk's FP64 orbital row reads, on the host:
for every pair of spin sizes each wave's eight columns lie inside the row of the
moved spin's padded coefficients, and a wave with orbitals of that spin reads
its own (the tile is the alpha spin's, the row length the moved spin's).  Points the
contraction reads: a walker group's last tile ends inside the basis scratch."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "qmcb_tiles.hpp"
using namespace qmcb;
int main() {
  int bad = 0;
  for (int up = 1; up <= 128; up++)
    for (int n = 1; n <= up; n++) {  // electrons of the moved spin
      const int NC = walk_tile(up), ldc = pad_orb(n);
      bad += up > NC || n > ldc || ldc % 16 != 0;
      for (int wave = 0; wave < NC / 16; wave++)
        for (int half = 0; half < 2; half++) {
          const int own = half * (NC / 2) + 8 * wave, c = walk_row_cols(wave, half, NC, ldc);
          bad += c < 0 || c % 2 != 0 || c + 8 > ldc;  // inside the row, 16-byte aligned
          bad += own < n && c != own;                 // its own orbitals
        }
    }
  const long rows = 5 * 64;
  const long sizes[] = {1, 64, 8192, 16448, 65536, 100032};
  for (long W : sizes)
    for (long G = 1; G <= 8 && G <= W; G++) {
      const long ldp = (W + 63) / 64 * 64, first = W * (G - 1) / G, cnt = W - first;
      const long last = (rows - 1) * ldp + first + (cnt + 31) / 32 * 32 - 1;
      bad += last >= (long)x_elems(rows, ldp);
    }
  printf("%d\n", bad);
  return bad != 0;
}
"""


def test_walk_row_columns_stay_inside_the_row(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    r = subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I",
                        os.path.join(ROOT, "qmcbeaver_amd", "csrc"), str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
