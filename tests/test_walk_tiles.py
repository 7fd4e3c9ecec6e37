"""Ranges of device reads and the length of a walk launch, on the host.

* The device walk's FP64 orbital row loads every column of the alpha spin's tile
  from the moved spin's coefficients: for every pair of spin sizes its last
  element lies inside the array.
* The contraction reads whole tiles of points: a walker group's last one ends
  inside the basis scratch.
* A launch of the walk is at least a step and, unless one step is longer, at most
  a tenth of a second by its own estimate.
"""
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
      const long NC = walk_tile(up), ldc = pad_orb(n);
      bad += up > NC || n > ldc;
      for (long kpad = 32; kpad <= 320; kpad += 32)
        bad += (kpad - 1) * ldc + NC - 1 >= (long)coef_elems(kpad, up, n);
    }
  const long rows = 5 * 64;
  const long sizes[] = {1, 64, 8192, 16448, 65536, 100032};
  for (long W : sizes)
    for (long G = 1; G <= 8 && G <= W; G++) {
      const long ldp = (W + 63) / 64 * 64, first = W * (G - 1) / G, cnt = W - first;
      const long last = (rows - 1) * ldp + first + (cnt + 31) / 32 * 32 - 1;
      bad += last >= (long)x_elems(rows, ldp);
    }
  for (int n = 1; n <= 128; n++)
    for (long W = 1; W <= 1000000; W *= 10) {
      const long steps = walk_most_steps(n, W);
      bad += steps < 1 || (steps > 1 && steps * (10.0 + W * (16.0 + n * n / 128) / 1e3) > 1e5);
    }
  printf("%d\n", bad);
  return bad != 0;
}
"""


def test_reads_stay_inside_their_arrays(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    r = subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I",
                        os.path.join(ROOT, "qmcbeaver_amd", "csrc"), str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
