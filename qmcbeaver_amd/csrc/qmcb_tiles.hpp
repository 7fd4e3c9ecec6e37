// Orbital padding, the column tiles of the device walk and the columns its
// FP64 rows read (no device headers: a host program can check the ranges).
#pragma once

namespace qmcb {

// Padded orbital count of a spin, the row length of its coefficients.
constexpr int pad_orb(int n) {
  return n > 64 ? (n + 127) / 128 * 128 : n > 32 ? 64 : n > 16 ? 32 : 16;
}

// Elements of the basis scratch, `rows` rows (functions times components) of ldp
// points.  A contraction launch reads whole tiles of up to 32 points; those of
// a walker group start anywhere in a row, so that the last group's last tile
// may end past the last row.
constexpr long kPointTile = 32;
constexpr unsigned long x_elems(long rows, long ldp) {
  return (unsigned long)(rows * ldp + kPointTile);
}

// Columns of walk_kernel's tile, by the alpha electrons.
constexpr int walk_tile(int n) {
  return n <= 16 ? 16 : n <= 32 ? 32 : n <= 64 ? 64 : n <= 96 ? 96 : 128;
}

// Elements of the padded coefficients [kpad][pad_orb(n)] of a spin's n orbitals.
// walk_kernel's FP64 row loads every column of the alpha spin's tile: for a beta
// spin padded to fewer orbitals those past a row are the next rows' (loaded and
// not used), and the last row's are the elements added here.  Loads bounded to
// the row cost the 32-column tile 1 to 3 % of a step.
constexpr unsigned long coef_elems(long kpad, int n_up, int n) {
  const int over = walk_tile(n_up) - pad_orb(n);
  return (unsigned long)(kpad * pad_orb(n) + (over > 0 ? over : 0));
}

// Most steps of one launch of walk_kernel, about a tenth of a second: other
// contexts' work on the card waits behind a launch.  A step of `walkers` walkers
// takes roughly 10 us and 16 + n^2 / 128 ns a walker (n electrons a spin; 8192
// walkers of 60 electrons, FP32 operands: 152 us, 196 by this; 3000 of 256,
// FP64: 390 and 442).  A cut costs the state's trip to memory and back, 0.2 ms
// for the latter.
constexpr int walk_most_steps(int n, long walkers) {
  const double us = 10.0 + 1e-3 * walkers * (16.0 + n * n / 128.0);
  return us < 1e5 ? (int)(1e5 / us) : 1;
}

}  // namespace qmcb
