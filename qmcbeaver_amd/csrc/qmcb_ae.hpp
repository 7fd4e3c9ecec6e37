// Proposal and decision of an all-electron move by one workgroup a walker, the
// same bits in whichever kernel they run (products are contracted explicitly).
#pragma once
#include "qmcb_kernels.hpp"

namespace qmcb {

constexpr int kAeT = 256;  // most threads of a workgroup, a thread an electron

// v[k] summed over the workgroup of NW waves (waves in order)
template <int NV, int NW>
__device__ __forceinline__ void block_sums(double (&v)[NV], double (*scratch)[NW]) {
  const int t = threadIdx.x;
  if constexpr (NW == 1) {
#pragma unroll
    for (int k = 0; k < NV; k++) v[k] = wave_sum(v[k]);
    return;
  }
#pragma unroll
  for (int k = 0; k < NV; k++) {
    const double s = wave_sum(v[k]);
    if ((t & 63) == 0) scratch[k][t >> 6] = s;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; k++) {
    double s = 0.0;
    for (int q = 0; q < NW; q++) s += scratch[k][q];
    v[k] = s;
  }
  __syncthreads();
}

// The accept draw of step `step` of walker w.
__device__ __forceinline__ double ae_uniform(const AeArgs &A, long step, int w) {
  const uint32_t s0 = (uint32_t)step, s1 = (uint32_t)((uint64_t)step >> 32);
  const u4 r = philox4x32(u4{s0, s1, (uint32_t)w, kAeTag - 1u}, (uint32_t)A.seed,
                          (uint32_t)(A.seed >> 32));
  return u01(r.x, r.y);
}

// Proposal x + tau f + chi of electron e, written over R with x kept in Rsave;
// |chi|^2 is returned.
__device__ __forceinline__ double ae_propose_electron(const AeArgs &A, long step, int w, int e,
                                                      const double x[3], const double f[3]) {
  const uint32_t s0 = (uint32_t)step, s1 = (uint32_t)((uint64_t)step >> 32);
  const double st = sqrt(A.tau), two_pi = 6.283185307179586;
  // counter (step, walker, tag): tags 0 and 1 are the single-electron
  // proposal's, kAeTag + e this electron's, kAeTag - 1 the accept draw
  const u4 r = philox4x32(u4{s0, s1, (uint32_t)w, kAeTag + (uint32_t)e}, (uint32_t)A.seed,
                          (uint32_t)(A.seed >> 32));
  const double u0 = u01(r.x, r.y), u1 = u01(r.y, r.z), u2 = u01(r.z, r.w), u3 = u01(r.w, r.x);
  const double r1 = sqrt(-2.0 * log(u0)), r2 = sqrt(-2.0 * log(u2));
  const double g[3] = {r1 * cos(two_pi * u1), r1 * sin(two_pi * u1), r2 * cos(two_pi * u3)};
  double *xo = A.R + ((long)w * A.N + e) * 3, *xs = A.Rsave + ((long)w * A.N + e) * 3;
  double sq = 0.0;
  for (int k = 0; k < 3; k++) {
    const double chi = st * g[k];
    xs[k] = x[k];
    xo[k] = __builtin_fma(st, g[k], __builtin_fma(A.tau, f[k], x[k]));
    sq = __builtin_fma(chi, chi, sq);
  }
  return sq;
}

// The proposal of step `step` of walker w (batch row b) by a workgroup, a thread
// an electron at x with drift f.
template <int NW>
__device__ __forceinline__ void ae_propose_block(const AeArgs &A, long step, int b, int w,
                                                 const double x[3], const double f[3],
                                                 double (*scratch)[NW]) {
  const int t = threadIdx.x;
  double sq[1] = {0.0};
  if (t < A.N) sq[0] = ae_propose_electron(A, step, w, t, x, f);
  block_sums(sq, scratch);
  if (t == 0) {
    A.fwd[w] = sq[0];
    A.unif[b] = ae_uniform(A, step, w);
  }
}

// A walker's record and accumulators, loaded together.
struct AeRecord {
  double logpsi, sgn, mr, fwd, el, unif, acc_el, acc_el2, acc_n, acc_prop_el, weight, acc_w;
  int age;
};
__device__ __forceinline__ AeRecord ae_record(const AeArgs &A, int b, int w) {
  AeRecord r;
  r.logpsi = A.logpsi[w];
  r.sgn = A.sgn[w];
  r.mr = A.mr[w];
  r.fwd = A.fwd[w];
  r.el = A.cur_el[w];
  r.unif = A.unif[b];
  r.acc_el = A.acc_el[w];
  r.acc_el2 = A.acc_el2[w];
  r.acc_n = A.acc_n[w];
  r.acc_prop_el = A.acc_prop_el[w];
  r.weight = A.mode == 2 ? A.weight[w] : 1.0;
  r.acc_w = A.mode == 2 ? A.acc_w[w] : 0.0;
  r.age = A.walk.age ? A.walk.age[w] : 0;
  return r;
}

// Metropolis decision of a proposal with the sums |modified drift|^2, |drift|^2
// and reverse Green's function over its electrons; the lane with `write` writes
// the walker's scalars and the observable sample.
__device__ __forceinline__ bool ae_decide(const AeArgs &A, const AeRecord &o, double msq, double gsq,
                                          double rev, double EL, double lp_new, double sg_new,
                                          bool singular, int b, int w, bool write) {
  const double mr_t = gsq > 0.0 ? sqrt(msq) / sqrt(gsq) : 1.0;
  const bool sing = singular || !isfinite(lp_new) || !isfinite(EL);
  double p = sing ? 0.0 : exp(__builtin_fma(2.0, lp_new - o.logpsi,
                                            -((rev - o.fwd) / (2.0 * A.tau))));
  if (!(p == p)) p = 0.0;
  else if (!sing) p = old_walker_boost(p, o.age, A.walk.old_walker);
  if (A.mode == 2 && sg_new * o.sgn < 0) p = 0.0;  // fixed node (QMCWalker.cpp:1641-1646)
  if (p > 1.0) p = 1.0;
  const bool accept = p > o.unif;
  if (!write) return accept;
  const int age_new = accept ? 0 : o.age + 1;
  if (accept) {
    A.logpsi[w] = lp_new;
    A.sgn[w] = sg_new;
    A.mr[w] = mr_t;
    A.cur_el[w] = EL;
  }
  const double el = accept ? EL : o.el;
  if (A.walk.age) A.walk.age[w] = age_new;
  double wt = 1.0;
  if (A.mode == 2) {
    // umrigar93_probability_weighted reweighting at every all-electron step
    // (UNR93 eq. 25): dW = exp(tau_eff (p (S' + S) / 2 + (1 - p) S))
    wt = o.weight;
    if (A.reweight) {
      double so_, st_;
      if (A.energy_mod) {
        so_ = __builtin_fma(A.e_est - o.el, o.mr, A.e_trial - A.e_est);
        st_ = __builtin_fma(A.e_est - EL, mr_t, A.e_trial - A.e_est);
      } else {
        so_ = A.e_trial - o.el;
        st_ = A.e_trial - EL;
      }
      if (!(p > 0.0)) st_ = 0.0;
      const double dW = exp(A.tau_eff * __builtin_fma(p * 0.5, so_ + st_, (1.0 - p) * so_));
      wt = reweight_walker(wt, dW, age_new, el, A.walk);
      A.weight[w] = wt;
    }
    A.acc_w[w] = o.acc_w + wt;
  }
  A.acc_el[w] = __builtin_fma(wt, el, o.acc_el);
  A.acc_el2[w] = __builtin_fma(wt * el, el, o.acc_el2);
  A.acc_n[w] = o.acc_n + (accept ? 1.0 : 0.0);
  A.acc_prop_el[w] = o.acc_prop_el + (sing ? 0.0 : EL);
  if (A.obs) {
    // estimator p E_L(R') + (1 - p) E_L(R) (QMCWalker.cpp:2096-2104)
    A.obs[3L * b] = p > 0.0 ? __builtin_fma(p, EL, (1.0 - p) * o.el) : o.el;
    A.obs[3L * b + 1] = wt;
    A.obs[3L * b + 2] = p;
  }
  return accept;
}

// The sums of ae_decide, a thread an electron: x the proposal, xs where it came
// from, d the modified drift there, g the drift.
__device__ __forceinline__ void ae_sums(const AeArgs &A, const double x[3], const double xs[3],
                                        const double d[3], const double g[3], double v[3]) {
  for (int k = 0; k < 3; k++) {
    v[0] = __builtin_fma(d[k], d[k], v[0]);
    v[1] = __builtin_fma(g[k], g[k], v[1]);
    const double tt = __builtin_fma(-A.tau, d[k], xs[k] - x[k]);
    v[2] = __builtin_fma(tt, tt, v[2]);
  }
}

}  // namespace qmcb
