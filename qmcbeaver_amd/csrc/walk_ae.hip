// walk_ae.hip -- all-electron importance-sampled moves of the device walk
// (the reference's default, one_e_per_iter 0): every electron of a walker
// moves at once, the whole evaluate runs at the proposal, and the move is
// accepted or the walker's record restored.
//
// Reference: QMCWalker::initializePropagation / moveElectronsImportanceSampling
// (QMCWalker.cpp:179-198, 343-398: R' = R + tau F(R) + sqrt(tau) xi for all
// electrons, forward G = (2 pi tau)^(-3N/2) exp(-sum |sqrt(tau) xi|^2 /
// (2 tau))), calculateReverseGreensFunctionImportanceSampling (:756-780:
// exp(-sum |R - R' - tau F(R')|^2 / (2 tau)) with the same prefactor),
// calculateMoveAcceptanceProbability / acceptOrRejectMove (:1578-1685),
// processPropagation (:200-266: on rejection the saved record is restored,
// :259-262; reweighting at every all-electron step, :226-228) and
// reweight_walker (:1060-1185).
//
// The walker's current record lives in `drift` (the modified drift F at R,
// all electrons), `logpsi`, `sgn`, `mr` (|modified drift| / |drift|, the
// umrigar93 energy modification's ratio) and cur_el.  A move writes R' over
// R (saving R in Rsave), the ordinary all-electron evaluate runs at R' and
// its batch-row outputs `prop` decide the move: accepted, `prop` becomes the
// record; rejected, R is restored and the record kept.  The Slater and
// Jastrow state of a rejected walker then describes R', which no
// all-electron move reads; the host re-evaluates every walker at R after its
// last step, so the resident state describes R between calls.
//
// These kernels are the first proposal and the first record of a call; between
// steps the evaluate's last kernel (finish.hip) does both, except where it is
// replayed from a captured graph or the wave function has several determinants.
#include "qmcb_ae.hpp"
#include "qmcb_kernels.hpp"

namespace qmcb {

// FT threads: a wave up to 64 electrons, the same sums (65536 walkers of 2
// electrons: 70 us a proposal, 104 with four waves)
template <int FT>
__global__ void __launch_bounds__(FT) ae_propose_kernel(AeArgs A, const int *walkers, int num) {
  __shared__ double scratch[1][FT / 64];
  const int b = blockIdx.x, t = threadIdx.x;
  if (b >= num) return;
  const int w = walkers ? walkers[b] : b;
  double x[3] = {0.0, 0.0, 0.0}, f[3] = {0.0, 0.0, 0.0};
  if (t < A.N)
    for (int k = 0; k < 3; k++) {
      x[k] = A.R[((long)w * A.N + t) * 3 + k];
      f[k] = A.drift[((long)w * A.N + t) * 3 + k];
    }
  ae_propose_block(A, A.step, b, w, x, f, scratch);
}

// Metropolis decision of the walkers from the outputs `prop`; mode 0: the
// outputs become the walker's record (an evaluate of its current positions).
template <int FT>
__global__ void __launch_bounds__(FT) ae_accept_kernel(AeArgs A, const int *walkers, int num) {
  __shared__ double scratch[3][FT / 64];
  const int b = blockIdx.x, t = threadIdx.x;
  if (b >= num) return;
  const int w = walkers ? walkers[b] : b, N = A.N;
  const qmcb_results &P = A.prop;
  const AeRecord rec = ae_record(A, b, w);
  double x[3], xs[3], d[3], g[3], v[3] = {0.0, 0.0, 0.0};
  if (t < N) {
    for (int k = 0; k < 3; k++) {
      x[k] = A.R[((long)w * N + t) * 3 + k];
      xs[k] = A.mode != 0 ? A.Rsave[((long)w * N + t) * 3 + k] : x[k];
      d[k] = P.mod_drift[((long)b * N + t) * 3 + k];
      g[k] = P.grad_lnpsi[((long)b * N + t) * 3 + k];
    }
    ae_sums(A, x, xs, d, g, v);
  }
  block_sums(v, scratch);
  const double EL = P.e_local[b], lp = P.log_psi[b], sg = P.sign_psi[b] < 0 ? -1.0 : 1.0;
  bool accept = true;
  if (A.mode != 0) {
    accept = ae_decide(A, rec, v[0], v[1], v[2], EL, lp, sg, P.singular[b] != 0, b, w, t == 0);
  } else if (t == 0) {
    A.logpsi[w] = lp;
    A.sgn[w] = sg;
    A.mr[w] = v[1] > 0.0 ? sqrt(v[0]) / sqrt(v[1]) : 1.0;
    A.cur_el[w] = EL;
  }
  if (t < N)
    for (int k = 0; k < 3; k++) {
      if (accept) A.drift[((long)w * N + t) * 3 + k] = d[k];
      else A.R[((long)w * N + t) * 3 + k] = xs[k];
    }
}

hipError_t launch_ae_propose(const AeArgs &a, const int *walkers, int num, hipStream_t st) {
  if (num <= 0) return hipSuccess;
  if (a.N > kAeT) return hipErrorInvalidValue;
  if (a.N <= 64)
    hipLaunchKernelGGL(ae_propose_kernel<64>, dim3(num), dim3(64), 0, st, a, walkers, num);
  else
    hipLaunchKernelGGL(ae_propose_kernel<kAeT>, dim3(num), dim3(kAeT), 0, st, a, walkers, num);
  return hipGetLastError();
}

hipError_t launch_ae_accept(const AeArgs &a, const int *walkers, int num, hipStream_t st) {
  if (num <= 0) return hipSuccess;
  if (a.N > kAeT) return hipErrorInvalidValue;
  if (a.N <= 64)
    hipLaunchKernelGGL(ae_accept_kernel<64>, dim3(num), dim3(64), 0, st, a, walkers, num);
  else
    hipLaunchKernelGGL(ae_accept_kernel<kAeT>, dim3(num), dim3(kAeT), 0, st, a, walkers, num);
  return hipGetLastError();
}

}  // namespace qmcb
