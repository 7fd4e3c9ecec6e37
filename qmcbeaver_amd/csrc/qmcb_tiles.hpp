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

// First of the eight consecutive coefficient columns that wave `wave` of a
// tile of NC columns reads for half `half` of its orbitals (NC / 16 waves).
// The tile is the alpha spin's: for a beta spin padded to fewer orbitals the
// columns past the row's ldc (a multiple of 16) do not exist, and a wave whose
// orbitals they would be reads the first ones and stores nothing.
constexpr int walk_row_cols(int wave, int half, int NC, int ldc) {
  const int c = half * (NC / 2) + 8 * wave;
  return c < ldc ? c : 0;
}

}  // namespace qmcb
