// orbitals.hip -- kernels (a) and (b) in one: the basis functions of a tile of
// points are formed chunk by chunk in LDS and contracted with the orbital
// coefficients by MFMA from there, so their values never reach memory.
//
// Reference: QMCBasisFunction::evaluateBasisFunctions (QMCBasisFunction.cpp:
// 287-403) and the five products Xw * C^T of QMCSlater::evaluate
// (QMCSlater.cpp:856-862).  The arithmetic is that of basis_kernel and
// orbital_gemm_kernel, the same bits: FP64 functions by shells, rounded to the
// operand type, contracted in ascending function order by 16x16x4 MFMA.
//
// For batches of at most a workgroup a CU, where the two kernels are chains of
// dependent loads on a few waves a SIMD: a workgroup holds a tile of
// 16 points and up to 4 orbital tiles of 16, and runs four stages on successive
// chunks of 32 functions, one barrier a chunk.  Waves 0-7 form the exponentials
// of one chunk's primitives (a lane: one primitive at one point) and the radial
// sums of the chunk before (one shell at one point; a shell that straddles two
// chunks is formed for both), waves 8-11 the functions of the one before that,
// and each further wave contracts the functions for one orbital tile, all five
// components (its coefficients come straight from L2, one chunk ahead).  The
// records the stages read come through LDS, loaded two chunks ahead.  The two
// spins of an all-electron evaluate share a launch where both fit (blockIdx.z):
// 128 walkers of 2 electrons 15 -> 7.5 us.
//
// Measured, FP32 operands: 1500 points x 75 orbitals x 804 functions 45 us
// (basis 27 + contraction 39 before), 512 x 100 x 1019 59 us (35 + 52).  In the
// latter a chunk takes 3900 cycles, of which the matrix cores are busy 1050 and a
// SIMD issues about 490 vector instructions, FP64 most of them and four cycles
// each: the two add up on this card rather than overlap, which is also why the
// kernel gains nothing once the batch fills the chip.  With FP64 operands 7
// registers are spilled.
#include <hip/hip_bf16.h>

#include <algorithm>

#include "qmcb_kernels.hpp"
#include "qmcb_mfma.hpp"

namespace qmcb {

namespace {
constexpr int kOrbExp = 8;    // waves of the exponentials and radial sums
constexpr int kOrbFun = 4;    // waves of the functions
constexpr int kOrbProd = kOrbExp + kOrbFun;
constexpr int kOrbTiles = 4;  // most orbital tiles of a workgroup
constexpr int kOrbPts = 16;   // points of a tile
typedef float f4 __attribute__((ext_vector_type(4)));

// N 16-byte words of a record array into LDS, through registers of NT threads
template <int N, int NT>
struct Staged {
  static constexpr int U = (N + NT - 1) / NT;
  f4 v[U];
  __device__ __forceinline__ void load(const void *src, int count, int t) {
#pragma unroll
    for (int u = 0; u < U; u++)
      v[u] = ((const f4 *)src)[min(t + u * NT, max(count - 1, 0))];
  }
  __device__ __forceinline__ void store(void *dst, int count, int t) const {
#pragma unroll
    for (int u = 0; u < U; u++)
      if (t + u * NT < count) ((f4 *)dst)[t + u * NT] = v[u];
  }
};
}  // namespace

template <typename TX, typename TO>
__global__ void __launch_bounds__(64 * (kOrbProd + kOrbTiles))
orbitals_kernel(DevSystem S, OrbSide side0, OrbSide side1, int nkc) {
  // blockIdx.z: the side, usually a spin
  const OrbSide &Q = blockIdx.z == 0 ? side0 : side1;
  const PointSet pts = Q.pts;
  const GemmOut o = Q.out;
  const TX *__restrict__ Ct = (const TX *)Q.Ct;
  const int ldc = Q.ldc, n_orb = Q.n_orb;
  typedef Mfma<TX> M;
  typedef typename M::acc_t acc_t;
  constexpr int KC = kOrbChunk, PT = kOrbPts;
  constexpr int VE = 16 / sizeof(TX);  // k steps of one 16-byte LDS read
  constexpr int NG = KC / (4 * VE);    // such reads of a chunk
  constexpr int CS = NG * 64 * VE;     // component stride in LDS
  typedef TX xv __attribute__((ext_vector_type(VE)));
  // functions: [component][k / (4 VE)][lane of the MFMA operand][k step]
  __shared__ TX xs[2][kComp * CS];
  __shared__ double exps[2][kOrbPrims][PT];
  __shared__ double sums[2][KC][3][PT];
  __shared__ OrbPrim prims[4][kOrbPrims];
  __shared__ OrbShell shells[4][KC];
  __shared__ OrbFn fns[2][KC];
  __shared__ int4 kcs[kOrbChunks];
  static_assert(sizeof(OrbFn) == 32 && sizeof(OrbShell) == 16 && sizeof(OrbPrim) == 48, "records");
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const long p0 = (long)blockIdx.x * PT;
  // beyond the smaller side
  if (p0 >= pts.P || 16 * (int)blockIdx.y * ((int)(blockDim.x >> 6) - kOrbProd) >= n_orb) return;
  const int steps = nkc + 3;

  for (int i = threadIdx.x; i < nkc; i += blockDim.x) kcs[i] = S.orb_kc[i];
  __syncthreads();
  if (wave < kOrbProd) {
    const int t = wave < kOrbExp ? threadIdx.x : threadIdx.x - 64 * kOrbExp;
    const int li = t % PT, q = t / PT;
    const long p = p0 + li;
    double r[3] = {0.0, 0.0, 0.0};
    if (p < pts.P) {
      const long row = p / pts.per_walker;
      const long wk = pts.walker_map ? pts.walker_map[row] : row;
      const double *x = pts.base + wk * pts.walker_stride + (p % pts.per_walker) * pts.point_stride;
      r[0] = x[0]; r[1] = x[1]; r[2] = x[2];
    }
    // the coordinates waited for here: left to its first use, in the loops, the
    // wait would also be for each iteration's record loads (800 cycles a chunk)
    asm volatile("" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]));
    if (wave < kOrbExp) {
      constexpr int HT = 64 * kOrbExp;
      Staged<3 * kOrbPrims, HT> sp;
      Staged<KC, HT> ss;
      int4 k0, k1, k2;  // shells [x, x + y), primitives [z, z + w) of chunks s - 1, s, s + 1
      auto load = [&](const int4 &k) {
        sp.load(S.orb_prim + k.z, 3 * k.w, t);
        ss.load(S.orb_sh + k.x, k.y, t);
      };
      auto store = [&](const int4 &k, int c) {
        sp.store(prims[c & 3], 3 * k.w, t);
        ss.store(shells[c & 3], k.y, t);
      };
      auto range = [&](int c) -> int4 {
        const int4 v = kcs[min(c, nkc - 1)];
        const bool in = c < nkc;
        return int4{__builtin_amdgcn_readfirstlane(v.x),
                    __builtin_amdgcn_readfirstlane(in ? v.y : 0),
                    __builtin_amdgcn_readfirstlane(v.z),
                    __builtin_amdgcn_readfirstlane(in ? v.w : 0)};
      };
      k0 = int4{0, 0, 0, 0};
      k1 = range(0);
      k2 = range(1);
      load(k1);
      store(k1, 0);
      load(k2);
      __syncthreads();
      for (int s = 0; s < steps; s++) {
        store(k2, s + 1);
        const int4 k3 = range(s + 2);
        load(k3);
        // exponentials of chunk s
#pragma unroll 2
        for (int i = q; i < k1.w; i += HT / PT) {
          const OrbPrim &f = prims[s & 3][i];
          const double dx = r[0] - f.c[0], dy = r[1] - f.c[1], dz = r[2] - f.c[2];
          const double rsq = __builtin_fma(dz, dz, __builtin_fma(dx, dx, dy * dy));
          exps[s & 1][i][li] = exp(-f.alpha * rsq);
        }
        // radial sums of chunk s - 1
        for (int sl = q; sl < k0.y; sl += HT / PT) {
          const OrbShell sh = shells[(s - 1) & 3][sl];
          const OrbPrim *f = &prims[(s - 1) & 3][sh.p0 - k0.z];
          const double *ex = &exps[(s - 1) & 1][sh.p0 - k0.z][li];
          double s0 = 0, s1 = 0, s2 = 0;
          constexpr int U = 6;
          for (int i0 = 0; i0 < sh.np; i0 += U) {  // six at a time, the missing ones zero
            double al[U], co[U], e[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
              const int i = min(i0 + u, sh.np - 1);
              al[u] = f[i].alpha;
              co[u] = f[i].coef;
              e[u] = ex[i * PT];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < U; u++) {
              const double c_ = i0 + u < sh.np ? co[u] : 0.0, ce = c_ * e[u];
              s0 = __builtin_fma(c_, e[u], s0);
              s1 = __builtin_fma(al[u], ce, s1);
              s2 = __builtin_fma(al[u] * al[u], ce, s2);
            }
          }
          double *w = &sums[(s - 1) & 1][sl][0][li];
          w[0] = s0;
          w[PT] = s1;
          w[2 * PT] = s2;
        }
        k0 = k1;
        k1 = k2;
        k2 = k3;
        __syncthreads();
      }
      return;
    }
    // functions of chunk s - 2
    constexpr int HT = 64 * kOrbFun;
    Staged<2 * KC, HT> sf;
    sf.load(S.orb_fn, 2 * KC, t);
    __syncthreads();
    for (int s = 0; s < steps; s++) {
      const int c = s - 2;
      if (c + 1 >= 0 && c + 1 < nkc) sf.store(fns[(c + 1) & 1], 2 * KC, t);
      if (c + 2 > 0 && c + 2 < nkc) sf.load(S.orb_fn + (long)(c + 2) * KC, 2 * KC, t);
      if (c >= 0 && c < nkc) {
#pragma unroll
        for (int u = 0; u < KC * PT / HT; u++) {
          const int fq = q + u * (HT / PT);
          const bool real = c * KC + fq < S.B;  // the padding's coefficients are zero
          const OrbFn f = fns[c & 1][fq];
          const double *sm = &sums[c & 1][f.sh][0][li];
          const double s0 = sm[0], s1 = sm[PT], s2 = sm[2 * PT];
          double d[3], sq[3], tw[3], px[3], dpx[3], lpx[3];
#pragma unroll
          for (int k = 0; k < 3; k++) {
            d[k] = r[k] - f.c[k];
            sq[k] = d[k] * d[k];
            tw[k] = 2.0 * d[k];
          }
          const double rsq = __builtin_fma(d[2], d[2], __builtin_fma(d[0], d[0], sq[1]));
#pragma unroll
          for (int k = 0; k < 3; k++) {
            const int pw = (f.pw >> (2 * k)) & 3;
            px[k] = pw == 0 ? 1.0 : (pw == 1 ? d[k] : sq[k]);
            dpx[k] = pw == 0 ? 0.0 : (pw == 1 ? 1.0 : tw[k]);
            lpx[k] = pw == 2 ? 2.0 : 0.0;
          }
          const double L = (double)((f.pw & 3) + ((f.pw >> 2) & 3) + ((f.pw >> 4) & 3));
          const double pxy = px[0] * px[1], P = pxy * px[2];
          const double val = P * s0;
          const double gx = __builtin_fma(s0, dpx[0] * px[1] * px[2], -(tw[0] * P * s1));
          const double gy = __builtin_fma(s0, px[0] * dpx[1] * px[2], -(tw[1] * P * s1));
          const double gz = __builtin_fma(s0, pxy * dpx[2], -(tw[2] * P * s1));
          const double lapP = __builtin_fma(
              pxy, lpx[2], __builtin_fma(px[2], lpx[0] * px[1], px[0] * lpx[1] * px[2]));
          const double lap =
              __builtin_fma(s2, 4.0 * rsq * P, __builtin_fma(s0, lapP, -((4.0 * L + 6.0) * P * s1)));
          TX *x = xs[c & 1] + (fq / (4 * VE)) * 64 * VE + ((fq & 3) * 16 + li) * VE + (fq >> 2) % VE;
          x[0] = real ? (TX)val : (TX)0;
          x[CS] = real ? (TX)gx : (TX)0;
          x[2 * CS] = real ? (TX)gy : (TX)0;
          x[3 * CS] = real ? (TX)gz : (TX)0;
          x[4 * CS] = real ? (TX)lap : (TX)0;
        }
      }
      __syncthreads();
    }
    return;
  }

  // contraction of chunk s - 3
  const int li = lane & 15, lk = lane >> 4;
  const int o0 = 16 * ((int)blockIdx.y * ((int)(blockDim.x >> 6) - kOrbProd) + wave - kOrbProd);
  const bool live = o0 < n_orb;
  acc_t acc[kComp];
#pragma unroll
  for (int c = 0; c < kComp; c++) acc[c] = acc_t{0, 0, 0, 0};
  const TX *cp = Ct + (long)lk * ldc + (live ? o0 : 0) + li;
  TX a[KC / 4], an[KC / 4];
#pragma unroll
  for (int s = 0; s < KC / 4; s++) a[s] = an[s] = cp[(long)(4 * s) * ldc];
  for (int s = 0; s < 4; s++) __syncthreads();
  for (int ch = 0; ch < nkc; ch++) {
    cp += (long)KC * ldc;
    if (ch + 1 < nkc) {
#pragma unroll
      for (int s = 0; s < KC / 4; s++) an[s] = cp[(long)(4 * s) * ldc];
    }
    if (live) {
      const TX *x = xs[ch & 1] + lane * VE;
#pragma unroll
      for (int g0 = 0; g0 < NG; g0 += 2) {  // two reads a component in flight
        xv b[2][kComp];
#pragma unroll
        for (int g = 0; g < 2; g++)
#pragma unroll
          for (int c = 0; c < kComp; c++)
            b[g][c] = *(const xv *)(x + c * CS + (g0 + g) * 64 * VE);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int g = 0; g < 2; g++)
#pragma unroll
          for (int s = 0; s < VE; s++)
#pragma unroll
            for (int c = 0; c < kComp; c++)
              acc[c] = M::run(a[(g0 + g) * VE + s], b[g][c][s], acc[c]);
      }
    }
#pragma unroll
    for (int s = 0; s < KC / 4; s++) a[s] = an[s];
    __syncthreads();
  }
  if (!live) return;
  const long p = p0 + li;
  if (p >= pts.P) return;
  struct alignas(4 * sizeof(TO)) Quad {
    TO v[4];
  };
  TO *out = (TO *)o.out;
  const long row = p / o.per_walker, pe = p % o.per_walker;
  const long wk = o.walker_map ? o.walker_map[row] : row;
  if (o.out_val) {
    // all electrons: FP64 values, and the four derivatives of an element
    // together (s_comp == 1)
    double *ov = o.out_val + wk * o.s_walker_val + pe * o.s_elec_val;
    TO *od = out + wk * o.s_walker + pe * o.s_elec;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int orb = o0 + M::row(lk, i);
      if (orb >= n_orb) continue;
      ov[(long)orb * o.s_orb_val] = (double)acc[0][i];
      Quad v;
#pragma unroll
      for (int c = 0; c < 4; c++) v.v[c] = (TO)acc[c + 1][i];
      *(Quad *)(od + (long)orb * o.s_orb) = v;
    }
  } else {
    // a row of contiguous orbitals a point; whole tiles, the padding with zeros
#pragma unroll
    for (int c = 0; c < kComp; c++) {
      TO *od = out + (long)c * o.s_comp + wk * o.s_walker + pe * o.s_elec + o0;
      if constexpr (M::row(0, 1) == 1) {
        Quad v;
#pragma unroll
        for (int i = 0; i < 4; i++) v.v[i] = (TO)acc[c][i];
        *(Quad *)(od + M::row(lk, 0)) = v;
      } else {
#pragma unroll
        for (int i = 0; i < 4; i++) od[M::row(lk, i)] = (TO)acc[c][i];
      }
    }
  }
}

// Workgroups of a launch.  One on each CU is the bound for this kernel
// (kOrbWorkgroups): up to it a step of the device walk is 1.05 to 1.23 times
// faster than with the two kernels (256 electrons x 500 walkers 165 -> 135 us,
// x 2000 at 250 workgroups 306 -> 271; 100 x 4000 at 250 156 -> 134; all-
// electron moves of 16 electrons x 500 walkers at 250 134 -> 111).  Beyond it
// the two kernels are as fast or faster: forms of this one with 32 points or 8
// orbital tiles a workgroup took 370 us at 342 workgroups (256 x 2731) against
// 303, and 5.6 ms for 1024 x 256 electrons at once against 5.8.
long orbitals_workgroups(long P, int n_orb) {
  return (P + kOrbPts - 1) / kOrbPts * ((n_orb + 16 * kOrbTiles - 1) / (16 * kOrbTiles));
}

template <typename TX, typename TO>
hipError_t launch_orbitals(const DevSystem &sys, const OrbSide &s0, const OrbSide *s1, int kpad,
                           hipStream_t st) {
  if (!s1 && (s0.pts.P <= 0 || s0.n_orb <= 0)) return hipSuccess;
  const int nkc = (sys.B + kOrbChunk - 1) / kOrbChunk;
  if (nkc * kOrbChunk > kpad || nkc > kOrbChunks) return hipErrorInvalidValue;
  long gx = 0;
  int gy = 0, cw = 0;
  for (const OrbSide *q : {&s0, s1}) {
    if (!q) continue;
    if (q->pts.P <= 0 || q->n_orb <= 0) return hipErrorInvalidValue;
    const int tiles = (q->n_orb + 15) / 16;
    const GemmOut &o = q->out;
    // whole orbital tiles in Ct; one of the two output forms
    const bool quads = o.s_elec % 4 == 0 && o.s_walker % 4 == 0 &&
                       (uintptr_t)o.out % (4 * sizeof(TO)) == 0;
    const bool form = o.out_val ? o.s_comp == 1 && o.s_orb % 4 == 0
                                : o.s_orb == 1 && o.s_comp % 4 == 0 && o.s_comp >= 16 * tiles;
    if (!quads || !form || 16 * tiles > q->ldc) return hipErrorInvalidValue;
    gx = std::max(gx, (q->pts.P + kOrbPts - 1) / kOrbPts);
    const int y = (tiles + kOrbTiles - 1) / kOrbTiles;
    gy = std::max(gy, y);
    cw = std::max(cw, (tiles + y - 1) / y);
  }
  hipLaunchKernelGGL((orbitals_kernel<TX, TO>), dim3((unsigned)gx, (unsigned)gy, s1 ? 2 : 1),
                     dim3(64 * (kOrbProd + cw)), 0, st, sys, s0, s1 ? *s1 : s0, nkc);
  return hipGetLastError();
}

#define QMCB_ORBITALS(TX, TO)                                                          \
  template hipError_t launch_orbitals<TX, TO>(const DevSystem &, const OrbSide &,      \
                                              const OrbSide *, int, hipStream_t);
QMCB_ORBITALS(double, double)
QMCB_ORBITALS(double, float)
QMCB_ORBITALS(float, float)
QMCB_ORBITALS(float, bf16s)

}  // namespace qmcb
