// Pade functions in LDS and their evaluation from there: the operations of
// pade_eval, the same bits.
#pragma once
#include "qmcb_common.hpp"

namespace qmcb {

// Pade functions packed in LDS: {n_num, n_den as two ints}, num[mn], den[md]
struct PadeShape {
  int mn, md;
  __host__ __device__ int stride() const { return 1 + mn + md; }
};
__device__ __forceinline__ void pade_general(const double *f, const PadeShape &ps, double r,
                                              double &u, double &du, double &d2u) {
  const long long cnt = __builtin_bit_cast(long long, f[0]);
  const int nn = (int)cnt, nd = (int)(cnt >> 32);
  const double *num = f + 1, *den = f + 1 + ps.mn;
  double a = 0.0, ap = 0.0, app = 0.0;
  if (nn > 0) {
    a = num[nn - 1];
    for (int i = nn - 2; i >= -1; i--) {
      const double c = i >= 0 ? num[i] : 0.0;
      app = app * r + ap;
      ap = ap * r + a;
      a = a * r + c;
    }
    app *= 2.0;
  }
  double b = 1.0, bp = 0.0, bpp = 0.0;
  if (nd > 0) {
    b = den[nd - 1];
    for (int i = nd - 2; i >= -1; i--) {
      const double c = i >= 0 ? den[i] : 1.0;
      bpp = bpp * r + bp;
      bp = bp * r + b;
      b = b * r + c;
    }
    bpp *= 2.0;
  }
  const double ib = 1.0 / b;
  u = a * ib;
  du = (ap - u * bp) * ib;
  d2u = (app - 2.0 * du * bp - u * bpp) * ib;
}
// u = a r / (1 + b r) with f = {a, b} (one term each), the same operations
__device__ __forceinline__ void pade_first(const double *f, double r, double &u, double &du,
                                           double &d2u) {
  const double ap = f[0], bp = f[1];
  const double b = __builtin_fma(bp, r, 1.0), ib = 1.0 / b;
  u = ap * r * ib;
  du = __builtin_fma(-u, bp, ap) * ib;
  d2u = -(2.0 * du * bp) * ib;
}

}  // namespace qmcb
