// finish.hip -- the end of an all-electron evaluate in one kernel: derivative
// traces of both spins, Jastrow factor and potential, assembly of Psi, its
// gradient and E_L, and, inside all-electron moves, the Metropolis decision and
// the next proposal.
//
// Reference: QMCSlater::calculate_DerivativeRatios (QMCSlater.cpp:731-762),
// QMCJastrow::evaluate (QMCJastrow.cpp:134-187), QMCJastrowElectronElectron::
// updateAll / collectForPair (QMCJastrowElectronElectron.cpp:56-298),
// QMCJastrowElectronNuclear::evaluate (QMCJastrowElectronNuclear.cpp:54-187),
// QMCPotential_Energy::calc_P_en/calc_P_ee (QMCPotential_Energy.cpp:242-333) and
// QMCSCFJastrow::calculate_Psi_quantities / calculate_E_Local
// (QMCSCFJastrow.cpp:196-282, QMCSCFJastrow.h:311-314).
//
// One workgroup per walker, of four waves, up to 16 electrons of one: of a small
// molecule four waves are mostly idle, and their LDS keeps all but three walkers
// off a CU (all-electron moves, us a step with four and with one: 2 electrons x
// 65536 walkers 1658 and 404, x 128 28.9 and 28.1; 10 x 16000 651 and 282).  For
// 32 electrons one wave took a twentieth longer at 128 walkers.
// Every sum that reaches a gradient keeps the order of a plain loop (orbitals
// ascending in a trace; nuclei, then partners ascending in a Jastrow gradient), so
// that gradients, and the walks that follow them, are bit for bit those of one
// thread an electron; sums that only reach energies and ln Psi are added in any
// order.
#include "qmcb_ae.hpp"
#include "qmcb_kernels.hpp"
#include "qmcb_pade.hpp"

namespace qmcb {

namespace {
constexpr int kFT = kAeT;   // threads
constexpr int kFN = 256;    // most electrons
constexpr int kTile = 64;   // particles of a pair tile
constexpr int kNuc = 40;    // nuclei of a tile (three workgroups' LDS on a CU)
constexpr int kLd = kTile + 1;
constexpr int kSmall = 16;  // most electrons (and nuclei of a tile) of the one-wave form

template <typename TS>
__device__ __forceinline__ double ldd(const TS *p) { return (double)*p; }

struct JastrowLds {
  static constexpr int kElectrons = kFN, kNuclei = kNuc;
  double x[kFN * 3];        // positions
  double g[3][kFN];         // Jastrow gradient
  double w[kTile * kLd];    // u'/r of a tile's pairs
  double ee[3][2];          // one-term Pade functions of the electron pair types
  double en[2][kNuc][2];   // ... and of a tile's nuclei, by spin
  double nuc[kNuc * 3], z[kNuc];
};

// the one-wave form's: 6 KB
struct SmallLds {
  static constexpr int kElectrons = kSmall, kNuclei = kSmall;
  double x[kSmall * 3], g[3][kSmall];
  double w[kSmall * (kSmall + 1)];
  double ee[3][2], en[2][kSmall][2];
  double nuc[kSmall * 3], z[kSmall];
};
template <int FT>
using FinishLds = std::conditional_t<FT == 64, SmallLds, JastrowLds>;

// Squared distance, the products contracted as in a plain loop.
__device__ __forceinline__ double dist2(const double *a, const double *b) {
  const double dx = a[0] - b[0], dy = a[1] - b[1], dz = a[2] - b[2];
  return __builtin_fma(dz, dz, __builtin_fma(dx, dx, dy * dy));
}

// Jastrow gradient of all electrons into L.g and, by thread, shares of U, its
// Laplacian, V_ee and V_en (v[0..3]).  L.x holds the positions.  ONE: every Pade
// function has one term in each polynomial (they come through LDS).
//
// A tile holds u'/r of up to 64 x 64 pairs, each formed once, by all threads (a
// thread an electron formed it twice with N of 256 threads busy: 37 us for 700
// walkers of 50 electrons, about 6 now; 365 us for 1024 of 256).
// Then a wave adds one coordinate of 64 gradients, partners ascending; tiles
// run by rows, the lower triangle's, whose mirror image is the partner rows'
// next block, so every gradient meets its partners in ascending order.
template <bool ONE>
__device__ __forceinline__ void jastrow_block(const DevSystem &S, JastrowLds &L, double v[4]) {
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int N = S.N, nn = S.nn, nu = S.n[0];
  for (int i = t; i < N; i += kFT) L.g[0][i] = L.g[1][i] = L.g[2][i] = 0.0;
  if (ONE && t < 3) {
    L.ee[t][0] = S.ee[t].num[0];
    L.ee[t][1] = S.ee[t].den[0];
  }
  // nuclei [a0, a0 + kNuc) with their Pade functions
  auto load_en = [&](int a0) {
    const int sp = t / 64, a = t % 64;
    if (a >= kNuc) return;
    if (sp < 3 && a0 + a < nn) L.nuc[3 * a + sp] = S.nuc_xyz[3 * (a0 + a) + sp];
    if (sp == 3 && a0 + a < nn) L.z[a] = S.nuc_z[a0 + a];
    if (ONE && sp < 2 && a0 + a < nn) {
      L.en[sp][a][0] = S.en[sp][a0 + a].num[0];
      L.en[sp][a][1] = S.en[sp][a0 + a].den[0];
    }
  };
  if (nn <= kNuc) load_en(0);
  // one coordinate of rows [r0, r0 + nr) gains `nc` partners at px, the pair's
  // value at w[row * sr + partner * sc]
  auto add = [&](int k, int r0, int nr, const double *px, int nc, int sr, int sc) {
    if (lane >= nr) return;
    double g = L.g[k][r0 + lane];
    const double xr = L.x[3 * (r0 + lane) + k], *w = L.w + lane * sr;
#pragma unroll 8
    for (int c = 0; c < nc; c++) g = __builtin_fma(w[c * sc], xr - px[3 * c + k], g);
    L.g[k][r0 + lane] = g;
  };
  for (int i0 = 0; i0 < N; i0 += kTile) {
    const int nr = min(kTile, N - i0);
    // nuclei
    for (int a0 = 0; a0 < nn; a0 += kNuc) {
      const int na = min(kNuc, nn - a0);
      __syncthreads();
      if (nn > kNuc) {
        load_en(a0);
        __syncthreads();
      }
      if (lane < nr) {
        const int i = i0 + lane, sp = i < nu ? 0 : 1;
        for (int a = wave; a < na; a += kFT / 64) {
          const double r = sqrt(dist2(L.x + 3 * i, L.nuc + 3 * a)), ir = 1.0 / r;
          double u, du, d2u;
          if constexpr (ONE) pade_first(L.en[sp][a], r, u, du, d2u);
          else pade_eval(S.en[sp][a0 + a], r, u, du, d2u);
          v[0] += u;
          v[1] += 2.0 * ir * du + d2u;
          v[3] -= L.z[a] * ir;
          L.w[lane * kLd + a] = du * ir;
        }
      }
      __syncthreads();
      if (wave < 3) add(wave, i0, nr, L.nuc, na, kLd, 1);
    }
    // electrons
    for (int j0 = 0; j0 <= i0; j0 += kTile) {
      const bool diag = j0 == i0;
      const int nc = min(kTile, N - j0);
      __syncthreads();
      auto pair = [&](int r, int c) {  // i = i0 + r > j = j0 + c
        const int i = i0 + r, j = j0 + c;
        const double d = sqrt(dist2(L.x + 3 * i, L.x + 3 * j)), ir = 1.0 / d;
        double u, du, d2u;
        if constexpr (ONE) pade_first(L.ee[ee_type(i, j, nu)], d, u, du, d2u);
        else pade_eval(S.ee[ee_type(i, j, nu)], d, u, du, d2u);
        v[0] += u;
        v[1] += 2.0 * (2.0 * ir * du + d2u);
        v[2] += ir;
        const double w = du * ir;
        L.w[r * kLd + c] = w;
        if (diag) L.w[c * kLd + r] = w;
      };
      if (diag) {
        // rows a and nr - 1 - a together hold nr - 1 pairs
        for (int a = wave; 2 * a < nr; a += kFT / 64) {
          const int b = nr - 1 - a;
          const bool up = lane < a;
          if (up || (b != a && lane - a < b)) pair(up ? a : b, up ? lane : lane - a);
          if (lane == 63) L.w[a * kLd + a] = L.w[b * kLd + b] = 0.0;
        }
      } else {
        for (int r = wave; r < nr; r += kFT / 64) pair(r, lane);  // a full block of partners
      }
      __syncthreads();
      for (int q = wave; q < (diag ? 3 : 6); q += kFT / 64) {
        if (q < 3) add(q, i0, nr, L.x + 3 * j0, nc, kLd, 1);
        else add(q - 3, j0, nc, L.x + 3 * i0, nr, 1, kLd);
      }
    }
  }
  __syncthreads();
}

// The same for up to kSmall electrons by one wave: a lane a pair, then a lane a
// coordinate of an electron, partners ascending.
template <bool ONE>
__device__ __forceinline__ void jastrow_block(const DevSystem &S, SmallLds &L, double v[4]) {
  constexpr int LD = kSmall + 1;
  const int t = threadIdx.x, N = S.N, nn = S.nn, nu = S.n[0];
  const int k = t / kSmall, r = t % kSmall;  // coordinate k < 3 of electron r
  auto add = [&](const double *px, int nc) {
    if (k >= 3 || r >= N) return;
    double g = L.g[k][r];
    const double xr = L.x[3 * r + k];
    for (int c = 0; c < nc; c++) g = __builtin_fma(L.w[r * LD + c], xr - px[3 * c + k], g);
    L.g[k][r] = g;
  };
  if (k < 3) L.g[k][r] = 0.0;
  if (ONE && t < 3) {
    L.ee[t][0] = S.ee[t].num[0];
    L.ee[t][1] = S.ee[t].den[0];
  }
  for (int a0 = 0; a0 < nn; a0 += kSmall) {
    const int na = min(kSmall, nn - a0);
    __syncthreads();
    if (t < 3 * na) L.nuc[t] = S.nuc_xyz[3 * a0 + t];
    if (t < na) L.z[t] = S.nuc_z[a0 + t];
    if (ONE && k < 2 && r < na) {
      L.en[k][r][0] = S.en[k][a0 + r].num[0];
      L.en[k][r][1] = S.en[k][a0 + r].den[0];
    }
    __syncthreads();
    for (int q = t; q < N * na; q += 64) {
      const int i = q / na, a = q % na, sp = i < nu ? 0 : 1;
      const double d = sqrt(dist2(L.x + 3 * i, L.nuc + 3 * a)), ir = 1.0 / d;
      double u, du, d2u;
      if constexpr (ONE) pade_first(L.en[sp][a], d, u, du, d2u);
      else pade_eval(S.en[sp][a0 + a], d, u, du, d2u);
      v[0] += u;
      v[1] += 2.0 * ir * du + d2u;
      v[3] -= L.z[a] * ir;
      L.w[i * LD + a] = du * ir;
    }
    __syncthreads();
    add(L.nuc, na);
  }
  __syncthreads();
  if (t < N) L.w[t * LD + t] = 0.0;
  // rows a and N - 1 - a together hold N - 1 pairs
  for (int q = t; q < (N + 1) / 2 * (N - 1); q += 64) {
    const int a = q / (N - 1), l = q % (N - 1), b = N - 1 - a;
    if (l >= a && b == a) continue;
    const int i = l < a ? a : b, j = l < a ? l : l - a;
    const double d = sqrt(dist2(L.x + 3 * i, L.x + 3 * j)), ir = 1.0 / d;
    double u, du, d2u;
    if constexpr (ONE) pade_first(L.ee[ee_type(i, j, nu)], d, u, du, d2u);
    else pade_eval(S.ee[ee_type(i, j, nu)], d, u, du, d2u);
    v[0] += u;
    v[1] += 2.0 * (2.0 * ir * du + d2u);
    v[2] += ir;
    L.w[i * LD + j] = L.w[j * LD + i] = du * ir;
  }
  __syncthreads();
  add(L.x, N);
  __syncthreads();
}

}  // namespace

// all-electron Jastrow and potential alone (several determinants)
template <bool ONE, int FT>
__global__ void __launch_bounds__(FT)
jastrow_all_kernel(JastrowArgs A, const int *walkers, int num) {
  __shared__ FinishLds<FT> L;
  __shared__ double scratch[4][FT / 64];
  const int b = blockIdx.x, t = threadIdx.x;
  if (b >= num) return;
  const int w = walkers ? walkers[b] : b, N = A.sys.N;
  for (int i = t; i < 3 * N; i += FT) L.x[i] = A.R[(long)w * N * 3 + i];
  __syncthreads();
  double v[4] = {0.0, 0.0, 0.0, 0.0};
  jastrow_block<ONE>(A.sys, L, v);
  block_sums(v, scratch);
  for (int i = t; i < 3 * N; i += FT) A.Ux[(long)w * N * 3 + i] = L.g[i % 3][i / 3];
  if (t == 0) {
    A.U[w] = v[0];
    A.Uxx[w] = v[1];
    A.Vee[w] = v[2];
    A.Ven[w] = v[3];
  }
}

hipError_t launch_jastrow_all(const JastrowArgs &a, bool pade_one, const int *walkers, int num,
                              hipStream_t st) {
  if (num <= 0) return hipSuccess;
  if (a.sys.N > kFN) return hipErrorInvalidValue;
  auto launch = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, dim3(num), dim3(threads), 0, st, a, walkers, num);
    return hipGetLastError();
  };
  if (a.sys.N <= kSmall)
    return pade_one ? launch(jastrow_all_kernel<true, 64>, 64) : launch(jastrow_all_kernel<false, 64>, 64);
  return pade_one ? launch(jastrow_all_kernel<true, kFT>, kFT) : launch(jastrow_all_kernel<false, kFT>, kFT);
}

// In place of two trace launches, Jastrow, assembly, decision and proposal: 700
// walkers of 50 electrons 76 -> 40 us a step, 128 of 2 electrons 31 -> 15, an
// evaluate of 1024 x 256 electrons 587 -> 390, of which the traces' inverse and
// derivatives are 180 at the copy rate.
//
// What a small walker spends its time on here is loads in a row (2 electrons:
// waits are 78 % of the waves' cycles), so everything that is known at the start
// is loaded there: the record of the move, and by electron (a thread each) the
// saved position and the drift it came from.
template <typename TS, bool ONE, int FT>
__global__ void __launch_bounds__(FT) finish_kernel(FinishArgs F, const int *walkers, int num) {
  typedef FinishLds<FT> Lds;
  static_assert(Lds::kElectrons <= FT, "a thread an electron");
  __shared__ Lds L;
  __shared__ double gs[Lds::kElectrons * 3];  // Slater gradient
  __shared__ double scratch[8][FT / 64];
  const int b = blockIdx.x, t = threadIdx.x;
  if (b >= num) return;
  const AssembleArgs &A = F.a;
  const DevSystem &S = A.sys;
  const int w = walkers ? walkers[b] : b;
  const int N = S.N, nu = S.n[0];
  const double *Rw = A.R + (long)w * N * 3;
  for (int i = t; i < 3 * N; i += FT) L.x[i] = Rw[i];
  double logdet = 0.0, sgn = 1.0;
  bool sp_sing[2] = {false, false};
#pragma unroll
  for (int sp = 0; sp < 2; sp++) {
    if (S.n[sp] == 0) continue;
    sp_sing[sp] = A.s[sp].singular[w] != 0;
    logdet += A.s[sp].logdet[w];
    sgn *= A.s[sp].sgn[w];
  }
  AeRecord rec{};
  double xs[3] = {0.0, 0.0, 0.0}, fo[3] = {0.0, 0.0, 0.0};
  if (F.move) {
    rec = ae_record(F.ae, b, w);
    if (t < N)
#pragma unroll
      for (int k = 0; k < 3; k++) {
        xs[k] = F.ae.Rsave[((long)w * N + t) * 3 + k];
        fo[k] = F.ae.drift[((long)w * N + t) * 3 + k];
      }
  }
  // ---- traces: a lane per (electron, derivative component), orbitals ascending.
  // Memory bound at 128 electrons a spin (inverse and derivatives read once);
  // with four lanes an electron short rows keep the loads of 25-electron spins
  // in flight as well.  A singular walker keeps its resident gradient.
  double lap[2] = {0.0, 0.0};
  for (int i = t; i < 4 * N; i += FT) {
    const bool dn = i >= 4 * nu;
    const int n = dn ? S.n[1] : nu, e0 = dn ? nu : 0;
    const int q = i - 4 * e0, e = q >> 2, k = q & 3;
    const double *inv = (dn ? A.s[1].inv : A.s[0].inv) + (long)w * n * n + e;
    const TS *dm = (const TS *)(dn ? A.s[1].dmat : A.s[0].dmat) + (long)w * kDer * n * n + q;
    double g = 0.0;
#pragma unroll 8
    for (int o = 0; o < n; o++) g = __builtin_fma(ldd(dm + (long)o * 4 * n), inv[(long)o * n], g);
    if (k == 3) {
      if (dn) lap[1] += g;
      else lap[0] += g;
    } else {
      double *gp = (dn ? A.s[1].gradPR : A.s[0].gradPR) + ((long)w * n + e) * 3 + k;
      if (dn ? sp_sing[1] : sp_sing[0]) g = *gp;
      else *gp = g;
      gs[3 * (e0 + e) + k] = g;
    }
  }
  __syncthreads();
  // U, its Laplacian, V_ee, V_en, the two traces; Laplacian cross terms, |grad|^2
  double v[8] = {0.0, 0.0, 0.0, 0.0, lap[0], lap[1], 0.0, 0.0};
  jastrow_block<ONE>(S, L, v);
  // ---- assembly, a thread an electron
  double g[3] = {0.0, 0.0, 0.0};
  if (t < N) {
    double *ux = F.Ux + ((long)w * N + t) * 3;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const double u = L.g[k][t], gp = gs[3 * t + k];
      ux[k] = u;
      g[k] = gp + u;
      v[6] += u * gp * 2.0;
      v[6] += u * u;
      v[7] += g[k] * g[k];
    }
    if (A.out.grad_lnpsi) {
      double *o = A.out.grad_lnpsi + ((long)b * N + t) * 3;
      o[0] = g[0]; o[1] = g[1]; o[2] = g[2];
    }
  }
  block_sums(v, scratch);
  bool sing = false;
  double lapR = v[1] + v[6];
#pragma unroll
  for (int sp = 0; sp < 2; sp++) {
    if (S.n[sp] == 0) continue;
    sing = sing || sp_sing[sp];
    lapR += sp_sing[sp] ? A.s[sp].lapPR[w] : v[4 + sp];
  }
  if (!(v[7] > 0.0) || !isfinite(v[7])) sing = true;
  double d[3] = {0.0, 0.0, 0.0};  // modified drift
  if (A.out.mod_drift && t < N) {
    double f = 1.0;
    if (A.drift_mod == QMCB_DRIFT_UMRIGAR93_EQUAL)
      f = (-1.0 + sqrt(1.0 + 2 * A.umrigar_a * v[7] * A.dt)) / (A.umrigar_a * v[7] * A.dt);
    if (A.drift_mod == QMCB_DRIFT_UMRIGAR93_UNEQUAL) {
      const double x[3] = {L.x[3 * t], L.x[3 * t + 1], L.x[3 * t + 2]};
      if (S.nn <= Lds::kNuclei) f = drift_factor_unequal(g, x, S.nn, L.nuc, L.z, A.dt);
      else f = drift_factor_unequal(g, x, S.nn, S.nuc_xyz, S.nuc_z, A.dt);
    }
    double *o = A.out.mod_drift + ((long)b * N + t) * 3;
#pragma unroll
    for (int k = 0; k < 3; k++) o[k] = d[k] = g[k] * f;
  }
  const double V = S.v_nn + v[2] + v[3];
  const double EL = -0.5 * lapR + V, lp = logdet + v[0];
  if (t == 0) {
    F.U[w] = v[0];
    F.Uxx[w] = v[1];
    F.Vee[w] = v[2];
    F.Ven[w] = v[3];
    for (int sp = 0; sp < 2; sp++)
      if (S.n[sp] > 0 && !sp_sing[sp]) A.s[sp].lapPR[w] = v[4 + sp];
    const qmcb_results &o = A.out;
    if (o.log_psi) o.log_psi[b] = lp;
    if (o.sign_psi) o.sign_psi[b] = (int8_t)(sgn < 0 ? -1 : 1);
    if (o.lap_ratio) o.lap_ratio[b] = lapR;
    if (o.e_local) o.e_local[b] = EL;
    if (o.kinetic) o.kinetic[b] = -0.5 * lapR;
    if (o.potential) o.potential[b] = V;
    if (o.v_ne) o.v_ne[b] = v[3];
    if (o.v_ee) o.v_ee[b] = v[2];
    if (o.det_ratio) o.det_ratio[b] = 1.0;
    if (o.jastrow_u) o.jastrow_u[b] = v[0];
    if (o.singular) o.singular[b] = sing ? 1 : 0;
    if (A.cur_el) A.cur_el[w] = EL;
    if (A.age) A.age[w] = 0;
  }
  if (!F.move) return;
  // ---- the move's decision, then the next proposal
  double s3[3] = {0.0, 0.0, 0.0};
  double x[3] = {0.0, 0.0, 0.0};
  if (t < N) {
#pragma unroll
    for (int k = 0; k < 3; k++) x[k] = L.x[3 * t + k];
    ae_sums(F.ae, x, xs, d, g, s3);
  }
  block_sums(s3, scratch);
  const bool accept = ae_decide(F.ae, rec, s3[0], s3[1], s3[2], EL, lp, sgn < 0 ? -1.0 : 1.0, sing,
                                b, w, t == 0);
  if (t < N) {
    double *xo = F.ae.R + ((long)w * N + t) * 3, *f = F.ae.drift + ((long)w * N + t) * 3;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      if (accept) {
        f[k] = d[k];
      } else {
        d[k] = fo[k];
        x[k] = xs[k];
        if (!F.propose) xo[k] = x[k];
      }
    }
  }
  if (F.propose) ae_propose_block(F.ae, F.ae.step + 1, b, w, x, d, scratch);
}

template <typename TS>
hipError_t launch_finish(const FinishArgs &f, const int *walkers, int num, hipStream_t st) {
  if (num <= 0) return hipSuccess;
  if (f.a.sys.N > kFN || f.a.s[0].ndet > 1 || f.a.s[0].occ || f.a.s[1].occ)
    return hipErrorInvalidValue;
  auto launch = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, dim3(num), dim3(threads), 0, st, f, walkers, num);
    return hipGetLastError();
  };
  if (f.a.sys.N <= kSmall)
    return f.pade_one ? launch(finish_kernel<TS, true, 64>, 64)
                      : launch(finish_kernel<TS, false, 64>, 64);
  return f.pade_one ? launch(finish_kernel<TS, true, kFT>, kFT)
                    : launch(finish_kernel<TS, false, kFT>, kFT);
}
template hipError_t launch_finish<double>(const FinishArgs &, const int *, int, hipStream_t);
template hipError_t launch_finish<float>(const FinishArgs &, const int *, int, hipStream_t);
template hipError_t launch_finish<bf16s>(const FinishArgs &, const int *, int, hipStream_t);

}  // namespace qmcb
