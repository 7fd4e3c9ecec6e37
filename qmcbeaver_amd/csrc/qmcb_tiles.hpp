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

}  // namespace qmcb
