// walk.hip -- a run of single-electron moves of the device walk in one launch:
// one workgroup carries one walker through consecutive steps (one determinant).
//
// Reference: the caller loop QMCWalker::initializePropagation /
// processPropagation (QMCWalker.cpp:179-282, 343-398, 756-780, 1060-1395,
// 1578-1685) around QMCSCFJastrow::evaluate (QMCSCFJastrow.cpp:91-472); the
// Slater part is QMCSlater's row replacement (QMCSlater.cpp:390-764).
//
// What bounds it: latency.  Step by step (proposal, basis, orbital GEMM,
// sm_move) a move of a small or medium molecule is 3-4 dependent launches,
// each a few microseconds of serial work; a move of a large one re-reads the
// walker's whole spin state (A^-1 and four derivative matrices) from HBM.  In
// one launch a step is a chain of LDS round trips, FP64 divisions, square
// roots, exponentials and wave sums of about 17 k cycles for two electrons and
// 32 k for 64 (waits are 35 and 42 % of them, vector instructions 46 and 33), with
// the moved spin's state on chip from move to move.  Time of a step, before (four launches) and now: 2 electrons x 128 walkers FP64 33.7
// and 8.8 us; 38 x 61 mixed 50.9 and 12.7; 122 x 50 mixed with cusps (DMC) 102
// and 25; 64 x 1024 FP64 73 and 16; 256 x 3000 FP64 692 and 390; 60 x 8192
// mixed 184 and 152.
//
// Mapping.  Columns c of the moved spin's A^-1 in NC columns (n <= NC), each
// in SL slices of consecutive rows: threads SL c + sl of a group hold the
// slice's elements (registers a[i]) and, with them, the derivative matrices'
// (d[i], with two or four groups of threads sharing the four components).
// Sums over a column are sums over the slice's rows, then over adjacent lanes
// (DPP, no LDS); an accepted move updates A^-1 in registers.  Thread e < N also
// holds electron e: position, Jastrow and determinant gradients, drift factor.
//   Derivatives in registers (FP32 operands; FP64 up to 32 columns): T1_k(c) =
//     sum_o d_k D(c,o) A^-1(o,c) and T2_k(c) = sum_o d_k D(c,o) A^-1(o,r) are
//     formed afresh at each move.
//   FP64 operands beyond: the moves run electron by electron, so the columns
//     r, r+1, ... of the next KB moves are known: one pass over the derivative
//     matrices forms T1 and T2 for all of them, and each accepted move updates
//     both by its rank-one term (T1 and T2 of the electrons replaced in the block
//     are formed from their new rows as stored).  The matrices are read once per
//     KB moves.
//     A run that ends inside a block leaves its sums in memory and the next one
//     goes on from them, so that a walk has the same bits however it is cut
//     into launches (calls, group tuning, other walkers' re-inversions).
//
// Steps of a move, seven workgroup barriers: proposal; exponentials (one
// primitive per thread) and the Jastrow pairs (thread e electron e, and
// nucleus e); basis functions, one per thread; the orbital row; w = v A^-1, T1
// and T2; ratio and new gradients; Green's functions; Metropolis.
// The row of FP32 operands is a chain of 4x4x1 matrix-core products, one
// function each in ascending order (32 orbitals x 5 components per wave):
// bit for bit the MFMA GEMM's sums, and 2.4 times the 16x16x4 form's rate
// where only five columns are used.  The row of FP64 operands is FMAs on a
// thread's four orbitals, sixteen slices of the functions.
// The random numbers of 64 steps are drawn at once, one step per lane.
// LDS reads are requested in groups ahead of a scheduling barrier: left to
// itself the compiler (with the flags that keep this loop's constants out of
// registers) waits on each one, 130 cycles a read.  The FP32 64-column tile
// spills 46 to 56 registers in the loop (112 to 120 bytes a lane); no other tile
// spills vector registers, and every one keeps 75 to 225 scalars in their lanes.
#include "qmcb_cusp.hpp"
#include "qmcb_kernels.hpp"
#include "qmcb_pade.hpp"
#include "qmcb_tiles.hpp"

namespace qmcb {

namespace {

// moves per pass over the derivative matrices where they are not held in
// registers (the 128-column tile's LDS takes four columns)
constexpr int walk_block(int NC) { return NC >= 128 ? 4 : 8; }

template <int CTRL>
__device__ __forceinline__ double quad_add(double v) { return v + dpp_f64<CTRL>(v); }
// sum over the four lanes of a quad; every lane gets it
__device__ __forceinline__ double quad_sum(double v) {
  v = quad_add<0xB1>(v);
  return quad_add<0x4E>(v);
}
// lane K of each quad to all its lanes
template <int K>
__device__ __forceinline__ double quad_bcast(double v) { return dpp_f64<K * 0x55>(v); }
// x + y of the lane 32 (16) away, after exchange: lanes of the lower half
// (even rows of 16) get both halves' (rows') x summed, the others their y
__device__ __forceinline__ double swap32_add(double x, double y) {
  const uint64_t a = __builtin_bit_cast(uint64_t, x), b = __builtin_bit_cast(uint64_t, y);
  const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)a, (uint32_t)b, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((uint32_t)(a >> 32), (uint32_t)(b >> 32), false, false);
  return __builtin_bit_cast(double, (uint64_t)hi[0] << 32 | lo[0]) +
         __builtin_bit_cast(double, (uint64_t)hi[1] << 32 | lo[1]);
}
__device__ __forceinline__ double swap16_add(double x, double y) {
  const uint64_t a = __builtin_bit_cast(uint64_t, x), b = __builtin_bit_cast(uint64_t, y);
  const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)a, (uint32_t)b, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)(a >> 32), (uint32_t)(b >> 32), false, false);
  return __builtin_bit_cast(double, (uint64_t)hi[0] << 32 | lo[0]) +
         __builtin_bit_cast(double, (uint64_t)hi[1] << 32 | lo[1]);
}
// of four values, the one of this lane's index q summed over the quad
__device__ __forceinline__ double quad_sum_own(double v0, double v1, double v2, double v3, int q) {
  // lanes 2j, 2j+1 exchange: even lanes keep (v0, v2), odd (v1, v3)
  const bool odd = q & 1;
  double a = odd ? v1 : v0, b = odd ? v3 : v2;
  const double sa = odd ? v0 : v1, sb = odd ? v2 : v3;
  a += dpp_f64<0xB1>(sa);
  b += dpp_f64<0xB1>(sb);
  const bool hi = q & 2;
  const double keep = hi ? b : a, send = hi ? a : b;
  return keep + dpp_f64<0x4E>(send);
}

// stored derivatives as the register copy holds them
template <typename TS> struct DerReg { typedef float T; };
template <> struct DerReg<double> { typedef double T; };

// KC (1, 2 or 4) adjacent components of an element
template <int KC, typename TS>
__device__ __forceinline__ void ld_der(const TS *p, typename DerReg<TS>::T d[KC]) {
  if constexpr (std::is_same<TS, bf16s>::value) {
    uint64_t q;
    if constexpr (KC == 4) q = *reinterpret_cast<const uint64_t *>(p);
    else if constexpr (KC == 2) q = *reinterpret_cast<const uint32_t *>(p);
    else q = *reinterpret_cast<const uint16_t *>(p);
#pragma unroll
    for (int k = 0; k < KC; k++)
      d[k] = __builtin_bit_cast(float, (uint32_t)((q >> (16 * k)) & 0xffffu) << 16);
  } else {
    constexpr int VE = sizeof(TS) == 8 ? 2 : KC;  // 16-byte loads, 8-byte for two floats
    typedef TS vec __attribute__((ext_vector_type(VE)));
#pragma unroll
    for (int h = 0; h < KC; h += VE) {
      const vec q = *reinterpret_cast<const vec *>(p + h);
#pragma unroll
      for (int k = 0; k < VE; k++) d[h + k] = q[k];
    }
  }
}
__device__ __forceinline__ void st_der(float *p, double x, double y, double z, double l) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  *reinterpret_cast<f4 *>(p) = f4{(float)x, (float)y, (float)z, (float)l};
}
__device__ __forceinline__ void st_der(double *p, double x, double y, double z, double l) {
  typedef double d2v __attribute__((ext_vector_type(2)));
  reinterpret_cast<d2v *>(p)[0] = d2v{x, y};
  reinterpret_cast<d2v *>(p)[1] = d2v{z, l};
}
__device__ __forceinline__ void st_der(bf16s *p, double x, double y, double z, double l) {
  *reinterpret_cast<uint64_t *>(p) = (uint64_t)bf16s(x).b | ((uint64_t)bf16s(y).b << 16) |
                                     ((uint64_t)bf16s(z).b << 32) | ((uint64_t)bf16s(l).b << 48);
}

// The basis values of one point in LDS.  FP64: five doubles a function (the
// sixteen functions a wave's row sum reads together fall in different banks).  FP32: [function / 4][8][function % 4], slots 0-4 the
// components, so that a lane reads four functions of its component at once.
template <typename TX> constexpr int kXWords = sizeof(TX) == 4 ? 8 : 5;  // words per function
template <typename TX>
__device__ __forceinline__ int x_at(int j) {
  return sizeof(TX) == 4 ? (j >> 2) * 32 + (j & 3) : j * 5;
}

// Threads of a workgroup and row slices of a column.  With FP32 operands the
// basis values are rounded to FP32, so a last-bit change of an FP64 sum can
// flip a rounding and be seen 2^-24 large: every sum that feeds a position or a
// stored row keeps sm_move_kernel's order (its slices, rows ascending within
// one, slices added in order; the tile being the alpha spin's, up to 16 beta
// electrons under more alpha ones have other slices than there).  FP64 operands
// take four slices throughout.
template <typename TX, int NC>
__host__ __device__ constexpr int walk_slices() {
  return sizeof(TX) == 8 || NC == 16 ? 4 : 2;
}
// groups of threads that share a column's four derivative components (each
// with the column of A^-1), FP32 operands: what keeps a thread near 256 registers
template <typename TX, int NC>
__host__ __device__ constexpr int walk_groups() {
  return sizeof(TX) == 8 || NC == 16 ? 1 : (NC == 32 ? 2 : 4);
}
template <typename TX, int NC>
__host__ __device__ constexpr int walk_threads() {
  return walk_groups<TX, NC>() * walk_slices<TX, NC>() * NC;
}
// whether the moved spin's derivative matrices are held in registers
template <typename TX>
__host__ __device__ constexpr bool der_in_reg(int NC) { return sizeof(TX) == 4 || NC <= 32; }
constexpr int kWalkWaves = 2;  // waves per SIMD the register allocation must allow

// drift_factor_near with the nucleus {x, y, z, Z} in LDS
__device__ __forceinline__ double drift_factor_lds(const double g[3], const double x[3],
                                                   const double *nuc, double dt) {
  double nv[3], dsq = 0.0;
#pragma unroll
  for (int k = 0; k < 3; k++) { nv[k] = x[k] - nuc[k]; dsq += nv[k] * nv[k]; }
  const double inr = 1.0 / sqrt(dsq);
  const double v2 = g[0] * g[0] + g[1] * g[1] + g[2] * g[2];
  const double iv = 1.0 / sqrt(v2);
  const double dotp = (nv[0] * g[0] + nv[1] * g[1] + nv[2] * g[2]) * inr * iv;
  const double Z = nuc[3];
  const double t = Z * Z * dsq;
  const double a = 0.5 * (1.0 + dotp) + t / (10.0 * (4.0 + t));
  const double f = (-1.0 + sqrt(1.0 + 2.0 * a * v2 * dt)) / (a * v2 * dt);
  return fabs(v2) < 1e-10 ? 1.0 : f;
}
// smallest value over the wave; every lane gets it
__device__ __forceinline__ double wave_min(double v) {
  v = fmin(v, dpp_f64<0xB1>(v));
  v = fmin(v, dpp_f64<0x4E>(v));
  v = fmin(v, dpp_f64<0x141>(v));
  v = fmin(v, dpp_f64<0x140>(v));
  return fmin(fmin(readlane_f64(v, 0), readlane_f64(v, 16)),
              fmin(readlane_f64(v, 32), readlane_f64(v, 48)));
}

// the quad's values added in lane order, ((0 + 1) + 2) + 3
__device__ __forceinline__ double quad_ordered(double v) {
  return ((quad_bcast<0>(v) + quad_bcast<1>(v)) + quad_bcast<2>(v)) + quad_bcast<3>(v);
}
__device__ __forceinline__ double quad_ordered_own(double v0, double v1, double v2, double v3,
                                                   int q) {
  const double a = quad_ordered(v0), b = quad_ordered(v1), c = quad_ordered(v2), d = quad_ordered(v3);
  return q == 0 ? a : (q == 1 ? b : (q == 2 ? c : d));
}

}  // namespace

template <typename TS, typename TX, int NC>
__global__ void
__attribute__((amdgpu_flat_work_group_size(walk_threads<TX, NC>(), walk_threads<TX, NC>()),
               amdgpu_waves_per_eu(kWalkWaves)))
walk_kernel(WalkArgs A, const int *walkers, int num) {
  constexpr int NT = walk_threads<TX, NC>(), NW = NT / 64, SL = walk_slices<TX, NC>(), KB = walk_block(NC);
  constexpr int RI = NC / SL;   // most rows of a slice
  constexpr int U8 = RI < 8 ? RI : 8;
  constexpr int NG = walk_groups<TX, NC>(), KC = 4 / NG;  // components of a group
  constexpr int NK = KC >= SL ? KC / SL : 1;  // components a lane of a column sums up
  constexpr bool ONE = KC < SL;               // one component, the same in both lanes
  constexpr bool F32 = sizeof(TX) == 4, RD = der_in_reg<TX>(NC);
  // stored derivatives narrower than the row they come from: a move's own traces
  // take the row as formed, every later one as stored, which in a block is T1 and
  // T2 of the electrons replaced
  constexpr bool NARROW = !RD && sizeof(TS) < sizeof(TX);
  typedef typename DerReg<TS>::T TD;
  const int b = blockIdx.x;
  if (b >= num) return;
  const int w = walkers ? walkers[b] : b;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int grp = NG > 1 ? wave / (NW / NG) : 0, c = t % (NC * SL) / SL, sl = t % SL;
  const int N = A.N, nu = A.n_up, nn = A.nn, B = A.B, kpad = A.kpad;  // FP32: a multiple of 48
  const PadeShape ps{A.pade_mn, A.pade_md};
  const int PS = ps.stride();
  const double tau = A.tau;
  const bool qf = A.drift_mod == QMCB_DRIFT_UMRIGAR93_UNEQUAL;

  __shared__ double s_col[2][NC];  // column r of A^-1 as [slice][RI], zero past a slice's rows
  __shared__ double s_v[kComp][NC];
  __shared__ double s_wv[NC];
  __shared__ double s_gq[4][NC];
  __shared__ double s_wj[7][NW], s_red[8][NW];
  __shared__ double s_draw[64][4];     // three normal deviates, one uniform
  __shared__ double s_xn[2][3], s_xo[2][3];
  __shared__ double s_new[4], s_held[4];  // the moved electron's T1 ratio, NARROW: of its stored row
  __shared__ double s_fix[KB][4];
  __shared__ double s_sc[17];  // thread 0's scalars, below
  __shared__ double s_psi[2][3];  // U and ln|det| of either spin, by step parity
  extern __shared__ __align__(16) unsigned char dyn[];
  TX *X = (TX *)dyn;                                     // basis values, x_words(kpad) values
  // tables, in the order of WalkArgs::tab
  double *s_prim = (double *)(X + (size_t)kpad * kXWords<TX>);  // [np]{exponent, coefficient}
  double *s_nuc = s_prim + 2 * A.np;                     // [nn]{x, y, z, Z}
  double *s_ee = s_nuc + 4 * nn;                         // [3][PS]
  double *s_en = s_ee + 3 * PS;                          // [2][nn][PS]
  uint64_t *s_fn = (uint64_t *)(s_en + 2 * nn * PS);     // [B] function records
  int *s_pa = (int *)(s_fn + B);                         // [np] atom of a primitive
  // scratch
  double *s_ex = (double *)(s_fn + B) + (A.np + 1) / 2;  // [np] exponentials
  double *s_rn = s_ex + A.np;                            // distance of the proposal to each nucleus
  double *s_blk = s_rn + nn;                             // not RD: [NC][KB] columns of A^-1
  double *s_vrow = s_blk + (RD ? 0 : NC * KB);           // not RD: [KB][NC][4] rows replaced

  // the tables as the host laid them out (formed here from the system's arrays, a
  // chain of dependent loads, they were half of a launch of one step)
  {
    typedef double d2v __attribute__((ext_vector_type(2)));
    for (int i = t; 2 * i < A.tab_len; i += NT) ((d2v *)s_prim)[i] = ((const d2v *)A.tab)[i];
  }
  for (int i = t; i < kpad * kXWords<TX>; i += NT) X[i] = (TX)0;
  for (int i = t; i < kComp * NC; i += NT) s_v[0][i] = 0.0;
  for (int i = t; i < 2 * NC; i += NT) s_col[0][i] = 0.0;

  // ---- walker state: thread e < N holds electron e's position, Jastrow and
  // determinant gradients, drift factor and nearest nucleus
  double Re[3] = {0, 0, 0}, Ue[3] = {0, 0, 0}, ge[3] = {0, 0, 0}, fo = 1.0;
  int cn = 0;
  const int esp = t < nu ? 0 : 1, ee_ = t - (esp ? nu : 0);  // electron t's spin, index in it
  if (t < N) {
    const long e = (long)w * N + t;
    const double *gp = A.s[esp].gradPR + ((long)w * (esp ? N - nu : nu) + ee_) * 3;
    for (int k = 0; k < 3; k++) {
      Re[k] = A.R[3 * e + k];
      Ue[k] = A.Ux[3 * e + k];
      ge[k] = gp[k];
    }
  }
  int age = A.walk.age ? A.walk.age[w] : 0;
  const bool sing0 = A.s[0].singular[w] != 0 || (N > nu && A.s[1].singular[w] != 0);
  // s_sc: 0 U, 1 Uxx, 2 Vee, 3 Ven, 4 E_L, 5-6 ln|det|, 7-8 sign, 9-10
  // Laplacian ratio per spin, 11 weight, 12-16 sums: w E_L, w E_L^2,
  // accepted, proposed E_L, w
  if (t == 0) {
    s_sc[0] = A.U[w]; s_sc[1] = A.Uxx[w]; s_sc[2] = A.Vee[w]; s_sc[3] = A.Ven[w];
    s_sc[4] = A.cur_el[w];
    for (int s = 0; s < 2; s++) {
      const bool some = s == 0 || N > nu;
      s_sc[5 + s] = some ? A.s[s].logdet[w] : 0.0;
      s_sc[7 + s] = some ? A.s[s].sgn[w] : 1.0;
      s_sc[9 + s] = some ? A.s[s].lapPR[w] : 0.0;
    }
    s_psi[0][0] = s_sc[0];
    s_psi[0][1] = s_sc[5];
    s_psi[0][2] = s_sc[6];
    s_sc[11] = A.mode == 2 ? A.weight[w] : 1.0;
    s_sc[12] = A.acc_el[w]; s_sc[13] = A.acc_el2[w]; s_sc[14] = A.acc_n[w];
    s_sc[15] = A.acc_prop_el[w];
    if (A.mode == 2) s_sc[16] = A.acc_w[w];
  }
  __syncthreads();
  if (qf && t < N) {
    double v[3];
    for (int k = 0; k < 3; k++) v[k] = ge[k] + Ue[k];
    cn = nearest_nucleus(Re, nn, s_nuc, 4);
    fo = drift_factor_lds(v, Re, s_nuc + 4 * cn, tau);
  }

  double a[RI];
  TD d[RD ? RI : 1][KC];
  double t1 = 0.0, G[RD ? 1 : KB];
  int cur = -1, blk_left = 0, nacc = 0, myacc = -1, n = 0, rows = 0, o_beg = 0, cl[2] = {0, 0};
  auto store_inv = [&](int sp) {
    if (c < n && grp == 0) {
      double *inv = A.s[sp].inv + (long)w * n * n;
#pragma unroll
      for (int i = 0; i < RI; i++)
        if (i < rows && o_beg + i < n) inv[(long)(o_beg + i) * n + c] = a[i];
    }
    if (t == 0) A.s[sp].dcount[w] = 0;
  };

  int obs_row = 0;
  int m_next = (int)(A.first_step % N);
  const double sqt = sqrt(tau);
  for (int sa = 0; sa < A.nsteps; sa += 64) {
    // the random numbers of the next 64 steps (propose_row's draws), one
    // step per lane of the first wave
    __syncthreads();
    if (t < 64) {
      const long st_ = A.first_step + sa + t;
      const uint32_t k0 = (uint32_t)A.seed, k1 = (uint32_t)(A.seed >> 32);
      double u[8];
      for (int cc = 0; cc < 2; cc++) {
        const u4 ctr = {(uint32_t)st_, (uint32_t)((uint64_t)st_ >> 32), (uint32_t)w, (uint32_t)cc};
        const u4 rr = philox4x32(ctr, k0, k1);
        u[4 * cc + 0] = u01(rr.x, rr.y);
        u[4 * cc + 1] = u01(rr.y, rr.z);
        u[4 * cc + 2] = u01(rr.z, rr.w);
        u[4 * cc + 3] = u01(rr.w, rr.x);
      }
      const double two_pi = 6.283185307179586;
      const double r1 = sqrt(-2.0 * log(u[0])), r2 = sqrt(-2.0 * log(u[2]));
      s_draw[t][0] = r1 * cos(two_pi * u[1]);
      s_draw[t][1] = r1 * sin(two_pi * u[1]);
      s_draw[t][2] = r2 * cos(two_pi * u[3]);
      s_draw[t][3] = u[4];
    }
    __syncthreads();
  for (int s = sa; s < min(sa + 64, A.nsteps); s++) {
    const int m = m_next;
    m_next = m + 1 == N ? 0 : m + 1;
    const int sp = m < nu ? 0 : 1;
    const int ss = sp ? nu : 0, r = m - ss;
    const int pb = s & 1;
    if (sp != cur) {
      if (cur >= 0) store_inv(cur);
      cur = sp;
      n = sp ? N - nu : nu;
      rows = (n + SL - 1) / SL;
      o_beg = sl * rows;
      blk_left = 0;
      if constexpr (!RD) {
        const int q = s == 0 ? A.s[sp].carried[w] : 0;
        if ((q >> 8) == m + 1) {  // go on in the block that the last run ended in
          const double *cb = A.carry + (long)w * (8 * KB * nu);
          const int n4 = 4 * n;
          blk_left = q & 15;
          nacc = (q >> 4) & 15;
          if (t < n4) {
            t1 = cb[t];
            myacc = (int)cb[n4 + t];
            for (int i = 0; i < nacc; i++) s_vrow[i * NT + t] = cb[(2 + i) * n4 + t];
#pragma unroll
            for (int j = 0; j < KB - 1; j++) G[j] = cb[(1 + KB + j) * n4 + t];
          }
        }
      }
      __syncthreads();
      for (int i = t; i < NC; i += NT)
        if (i >= n)
          for (int k = 0; k < kComp; k++) s_v[k][i] = 0.0;
      // places of column elements lane and lane + 64 in s_col
      cl[0] = lane / rows * RI + lane % rows;
      cl[1] = (lane + 64) / rows * RI + (lane + 64) % rows;
      const double *inv = A.s[sp].inv + (long)w * n * n;
      const TS *dm = (const TS *)A.s[sp].dmat + (long)w * kDer * n * n;
#pragma unroll
      for (int i = 0; i < RI; i++) {
        const int o = o_beg + i;
        const bool in = i < rows && o < n && c < n;
        a[i] = in ? inv[(long)o * n + c] : 0.0;
        if constexpr (RD) {
          TD z[KC];
#pragma unroll
          for (int k = 0; k < KC; k++) z[k] = (TD)0;
          if (in) ld_der<KC>(dm + 4 * ((long)o * n + c) + KC * grp, z);
#pragma unroll
          for (int k = 0; k < KC; k++) d[i][k] = z[k];
        }
      }
      const int dc = A.s[sp].dcount[w];
      for (int p = 0; p < dc; p++) {  // delayed terms left by other entry points
        const double *u = A.s[sp].ubuf + ((long)w * kDelay + p) * n;
        const double zc = c < n ? A.s[sp].zbuf[((long)w * kDelay + p) * n + c] : 0.0;
#pragma unroll
        for (int i = 0; i < RI; i++)
          if (i < rows && o_beg + i < n) a[i] -= u[o_beg + i] * zc;
      }
    }
    if constexpr (!RD) {
      if (blk_left == 0) {
        // one pass over the derivative matrices: T1 and T2 for the columns r .. r + KB - 1
        blk_left = min(KB, n - r);
        nacc = 0;
        myacc = -1;
        __syncthreads();
        if (c >= r && c < r + KB) {
#pragma unroll
          for (int i = 0; i < RI; i++)
            if (i < rows && o_beg + i < n) s_blk[(o_beg + i) * KB + c - r] = a[i];
        }
        if (r + KB > NC)  // columns past the tile have no owner
          for (int i = t; i < n * KB; i += NT)
            if (r + i % KB >= NC) s_blk[i] = 0.0;
        __syncthreads();
        const TS *dm = (const TS *)A.s[sp].dmat + (long)w * kDer * n * n + 4 * (long)min(c, n - 1);
        double p1[4] = {0, 0, 0, 0}, p2[KB][4];
#pragma unroll
        for (int j = 0; j < KB; j++)
#pragma unroll
          for (int k = 0; k < 4; k++) p2[j][k] = 0.0;
        constexpr int U = 2;
        TD nx[U][4];
#pragma unroll
        for (int u = 0; u < U; u++) ld_der<4>(dm + 4L * min(o_beg + u, n - 1) * n, nx[u]);
#pragma unroll
        for (int i0 = 0; i0 < RI; i0 += U) {
          if (i0 < rows) {
          TD cx[U][4];
#pragma unroll
          for (int u = 0; u < U; u++)
#pragma unroll
            for (int k = 0; k < 4; k++) cx[u][k] = nx[u][k];
          if (i0 + U < rows) {
#pragma unroll
            for (int u = 0; u < U; u++) ld_der<4>(dm + 4L * min(o_beg + i0 + U + u, n - 1) * n, nx[u]);
          }
#pragma unroll
          for (int u = 0; u < U; u++) {
            if (i0 + u < rows && o_beg + i0 + u < n) {
              const double *bc = s_blk + (o_beg + i0 + u) * KB;
#pragma unroll
              for (int k = 0; k < 4; k++) p1[k] += (double)cx[u][k] * a[i0 + u];
#pragma unroll
              for (int j = 0; j < KB; j++) {
                const double bj = bc[j];
#pragma unroll
                for (int k = 0; k < 4; k++) p2[j][k] += (double)cx[u][k] * bj;
              }
            }
          }
          }
        }
        t1 = quad_sum_own(p1[0], p1[1], p1[2], p1[3], sl);
#pragma unroll
        for (int j = 0; j < KB; j++) G[j] = quad_sum_own(p2[j][0], p2[j][1], p2[j][2], p2[j][3], sl);
      }
    }
    const double *draw = s_draw[s & 63];
    // ---- proposal by the moved electron's thread; column r by its owners
    if (t == m) {
#pragma unroll
      for (int k = 0; k < 3; k++) {
        double v = ge[k] + Ue[k];
        if (qf) v *= fo;
        s_xo[pb][k] = Re[k];
        s_xn[pb][k] = __builtin_fma(sqt, draw[k], __builtin_fma(tau, v, Re[k]));
      }
    }
    if (c == r && grp == 0) {
#pragma unroll
      for (int i = 0; i < RI; i++) s_col[pb][sl * RI + i] = a[i];
    }
    __syncthreads();
    const double xn[3] = {s_xn[pb][0], s_xn[pb][1], s_xn[pb][2]};
    const double xo[3] = {s_xo[pb][0], s_xo[pb][1], s_xo[pb][2]};
    const double *col = s_col[pb];
    // ---- exponentials of the basis at the proposal, one primitive per thread
    auto prim_exp = [&](int i) {
      const double *at = s_nuc + 4 * s_pa[i];
      const double d0 = xn[0] - at[0], d1 = xn[1] - at[1], d2 = xn[2] - at[2];
      const double rsq = d0 * d0 + d1 * d1 + d2 * d2;
      return exp(-s_prim[2 * i] * rsq);
    };
    for (int i = t; i < A.np; i += 2 * NT) {  // two independent ones at a time
      const int i2 = i + NT;
      const double e1 = prim_exp(i), e2 = prim_exp(min(i2, A.np - 1));
      s_ex[i] = e1;
      if (i2 < A.np) s_ex[i2] = e2;
    }
    // ---- Jastrow and potential at the proposal: thread t takes electron t's
    // pair with the moved electron at its new and old position, and nucleus t
    double js[7] = {0, 0, 0, 0, 0, 0, 0}, un_[3] = {0, 0, 0};
    auto jastrow = [&](auto pade) {
      // the pair and the first nucleus side by side (independent chains; both
      // are formed for a valid index and masked)
      const int a1 = min(t, nn - 1);
      double dn[3], dold[3], en_[3], eo_[3], rn2 = 0.0, ro2 = 0.0, sn2 = 0.0, so2 = 0.0;
#pragma unroll
      for (int k = 0; k < 3; k++) {
        dn[k] = xn[k] - Re[k]; rn2 += dn[k] * dn[k];
        dold[k] = xo[k] - Re[k]; ro2 += dold[k] * dold[k];
        en_[k] = xn[k] - s_nuc[4 * a1 + k]; sn2 += en_[k] * en_[k];
        eo_[k] = xo[k] - s_nuc[4 * a1 + k]; so2 += eo_[k] * eo_[k];
      }
      const double rn = sqrt(rn2), ro = sqrt(ro2), sn = sqrt(sn2), so = sqrt(so2);
      const double irn = 1.0 / rn, iro = 1.0 / ro, isn = 1.0 / sn, iso = 1.0 / so;
      const double *f = s_ee + ee_type(m, t, nu) * PS, *fe = s_en + (sp * nn + a1) * PS;
      double un, dun, d2un, uo, duo, d2uo, vn, dvn, d2vn, v_, dv_, d2v_;
      pade(f, rn, un, dun, d2un);
      pade(f, ro, uo, duo, d2uo);
      pade(fe, sn, vn, dvn, d2vn);
      pade(fe, so, v_, dv_, d2v_);
      if (t < N && t != m) {
        js[0] = un - uo;
        js[1] = 2.0 * (2.0 * irn * dun + d2un) - 2.0 * (2.0 * iro * duo + d2uo);
        js[2] = irn - iro;
        const double gn = dun * irn, go = duo * iro;
#pragma unroll
        for (int k = 0; k < 3; k++) {
          un_[k] = Ue[k] - gn * dn[k] + go * dold[k];
          js[4 + k] = gn * dn[k];
        }
      }
      if (t < nn) {
        s_rn[t] = sn;
        js[0] += vn - v_;
        js[1] += (2.0 * isn * dvn + d2vn) - (2.0 * iso * dv_ + d2v_);
        js[3] += s_nuc[4 * t + 3] * (iso - isn);
        const double gn = dvn * isn;
#pragma unroll
        for (int k = 0; k < 3; k++) js[4 + k] = __builtin_fma(gn, en_[k], js[4 + k]);
      }
      for (int a_ = t + NT; a_ < nn; a_ += NT) {
        double s2 = 0.0, t2 = 0.0;
#pragma unroll
        for (int k = 0; k < 3; k++) {
          en_[k] = xn[k] - s_nuc[4 * a_ + k]; s2 += en_[k] * en_[k];
          eo_[k] = xo[k] - s_nuc[4 * a_ + k]; t2 += eo_[k] * eo_[k];
        }
        const double r1 = sqrt(s2), r0 = sqrt(t2), i1 = 1.0 / r1, i0 = 1.0 / r0;
        s_rn[a_] = r1;
        const double *fa = s_en + (sp * nn + a_) * PS;
        pade(fa, r1, vn, dvn, d2vn);
        pade(fa, r0, v_, dv_, d2v_);
        js[0] += vn - v_;
        js[1] += (2.0 * i1 * dvn + d2vn) - (2.0 * i0 * dv_ + d2v_);
        js[3] += s_nuc[4 * a_ + 3] * (i0 - i1);
        const double gn = dvn * i1;
#pragma unroll
        for (int k = 0; k < 3; k++) js[4 + k] = __builtin_fma(gn, en_[k], js[4 + k]);
      }
    };
    if (64 * wave < max(N, nn)) {
      if (A.pade_one)
        jastrow([](const double *f, double x, double &u, double &du, double &d2u) {
          pade_first(f + 1, x, u, du, d2u);
        });
      else
        jastrow([&](const double *f, double x, double &u, double &du, double &d2u) {
          pade_general(f, ps, x, u, du, d2u);
        });
    }
#pragma unroll
    for (int k = 0; k < 7; k++) {
      const double sm = wave_sum(js[k]);
      if (lane == 0) s_wj[k][wave] = sm;
    }
    // ---- T2 of the electrons replaced earlier in this block, from their new rows
    if constexpr (!RD) {
      for (int i = wave; i < nacc; i += NW) {
        double f[4] = {0, 0, 0, 0};
#pragma unroll
        for (int h = 0; h < (NC + 63) / 64; h++)
          if (lane + 64 * h < n)
#pragma unroll
            for (int k = 0; k < 4; k++) f[k] += s_vrow[(i * NC + lane + 64 * h) * 4 + k] * col[cl[h]];
#pragma unroll
        for (int k = 0; k < 4; k++) f[k] = wave_sum(f[k]);
        if (lane == 0)
#pragma unroll
          for (int k = 0; k < 4; k++) s_fix[i][k] = f[k];
      }
    }
    __syncthreads();
    // FP32 row: the first coefficients are requested ahead of the barrier
    typedef float f4 __attribute__((ext_vector_type(4)));
    constexpr int UB = 4;  // groups of four functions per stage, three stages in flight
    const int og = 32 * wave;
    f4 cq[F32 ? 3 : 1][F32 ? UB : 1];
    const f4 *cw = (const f4 *)A.Cw[sp] + min(og + (lane & 31), NC - 1);
    auto row_load = [&](int g0, f4 *q) {
      const f4 *p = cw + g0 * NC;
#pragma unroll
      for (int u = 0; u < UB; u++) q[u] = p[u * NC];
    };
    // ---- basis functions, one per thread: radial sums, then the product rule
    for (int j = t; j < B; j += NT) {
      const uint64_t h = s_fn[j];
      const int np = (int)(h >> 6) & 0xFFFF, p0 = (int)(h >> 22) & 0x3FFFFF;
      const double *at = s_nuc + 4 * (int)(h >> 44);
      double dd[3];
#pragma unroll
      for (int k = 0; k < 3; k++) dd[k] = xn[k] - at[k];
      const double rsq = dd[0] * dd[0] + dd[1] * dd[1] + dd[2] * dd[2];
      double s0 = 0, s1 = 0, s2 = 0;
      for (int i0 = 0; i0 < np; i0 += 4) {  // four at a time, the missing ones zero
        double al[4], co[4], ex[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int i = p0 + min(i0 + u, np - 1);
          al[u] = s_prim[2 * i];
          co[u] = s_prim[2 * i + 1];
          ex[u] = s_ex[i];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const double c_ = i0 + u < np ? co[u] : 0.0, e = c_ * ex[u];
          s0 = __builtin_fma(c_, ex[u], s0);
          s1 = __builtin_fma(al[u], e, s1);
          s2 = __builtin_fma(al[u] * al[u], e, s2);
        }
      }
      const int pw[3] = {(int)h & 3, (int)(h >> 2) & 3, (int)(h >> 4) & 3};
      double px[3], dpx[3], lpx[3];
#pragma unroll
      for (int k = 0; k < 3; k++) {
        px[k] = pw[k] == 0 ? 1.0 : (pw[k] == 1 ? dd[k] : dd[k] * dd[k]);
        dpx[k] = pw[k] == 0 ? 0.0 : (pw[k] == 1 ? 1.0 : 2.0 * dd[k]);
        lpx[k] = pw[k] == 2 ? 2.0 : 0.0;
      }
      const double P = px[0] * px[1] * px[2];
      const double L = (double)(pw[0] + pw[1] + pw[2]);
      const double val = P * s0;
      const double gx = dpx[0] * px[1] * px[2] * s0 - 2.0 * dd[0] * P * s1;
      const double gy = px[0] * dpx[1] * px[2] * s0 - 2.0 * dd[1] * P * s1;
      const double gz = px[0] * px[1] * dpx[2] * s0 - 2.0 * dd[2] * P * s1;
      const double lapP = lpx[0] * px[1] * px[2] + px[0] * lpx[1] * px[2] + px[0] * px[1] * lpx[2];
      const double lap = lapP * s0 - (4.0 * L + 6.0) * P * s1 + 4.0 * rsq * P * s2;
      TX *o = X + x_at<TX>(j);
      constexpr int XS = F32 ? 4 : 1;  // distance of a function's components
      o[0] = (TX)val;
      o[XS] = (TX)gx;
      o[2 * XS] = (TX)gy;
      o[3 * XS] = (TX)gz;
      o[4 * XS] = (TX)lap;
    }
    if constexpr (F32)
      if (og < n) {
        row_load(0, cq[0]);
        row_load(UB, cq[1]);
        __builtin_amdgcn_sched_barrier(0);
      }
    __syncthreads();
    // ---- orbital row of the moved electron: v_k(o) = sum_b C(o,b) X_k(b)
    if constexpr (F32) {
      // wave g: orbitals 32g .. 32g + 31 by 4x4x1 outer products (16 blocks:
      // 0-7 the first four components, 8-15 the Laplacian), one function per
      // instruction in ascending order
      if (og < n) {
        const f4 *xp = (const f4 *)X + (lane < 32 ? (lane & 3) : 4 + (lane & 3));
        f4 acc = {0.f, 0.f, 0.f, 0.f};
        const int ng = kpad / 4;  // a multiple of the three stages
        f4 x[UB];
#pragma unroll
        for (int u = 0; u < UB; u++) x[u] = xp[8 * u];
        for (int g0 = 0; g0 < ng; g0 += 3 * UB) {
#pragma unroll
          for (int q = 0; q < 3; q++) {
            // the stage after next and the next basis values are requested
            // under this stage's sixteen products
            row_load(min(g0 + (q + 2) * UB, ng - UB), cq[(q + 2) % 3]);
            f4 y[UB];
            const int gn = min(g0 + (q + 1) * UB, ng - UB);
#pragma unroll
            for (int u = 0; u < UB; u++) y[u] = xp[8 * (gn + u)];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < UB; u++)
#pragma unroll
              for (int e = 0; e < 4; e++)
                acc = __builtin_amdgcn_mfma_f32_4x4x1f32(cq[q][u][e], x[u][e], acc, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < UB; u++) x[u] = y[u];
          }
        }
        const int k = lane < 32 ? lane & 3 : 4 + (lane & 3), o = og + 4 * ((lane >> 2) & 7);
        if (k < kComp)
#pragma unroll
          for (int i = 0; i < 4; i++)
            if (o + i < n) s_v[k][o + i] = (double)acc[i];
      }
    } else {
      // lane 4 ks + gl of wave v, g = 4v + gl: orbitals 2g, 2g + 1 and NC / 2 + 2g,
      // NC / 2 + 2g + 1 (four lanes load 64 consecutive bytes), functions
      // b = 16 i + ks; a basis value read from LDS serves four orbitals
      typedef double d2v __attribute__((ext_vector_type(2)));
      const int ks = lane >> 2, g2_ = 2 * (4 * wave + (lane & 3)), ldc = A.npad[sp];
      double f[4][kComp];
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int k = 0; k < kComp; k++) f[j][k] = 0.0;
      const double *cp = (const double *)A.Ct[sp] + (long)ks * ldc + g2_;
      const double *xp = (const double *)X + ks * kXWords<TX>;
      const int ni = kpad / 16;  // even
      constexpr int UD = 2;  // coefficient rows per stage, two stages in flight
      d2v ca[UD][2], cb[UD][2];
      auto load = [&](int i0, d2v (*q)[2]) {
#pragma unroll
        for (int u = 0; u < UD; u++) {
          const double *p = cp + 16L * (i0 + u) * ldc;
          q[u][0] = *(const d2v *)p;
          q[u][1] = *(const d2v *)(p + NC / 2);  // to column NC - 1 (coef_elems)
        }
      };
      auto mac = [&](int i0, const d2v (*q)[2]) {
        double x[UD][kComp];
#pragma unroll
        for (int u = 0; u < UD; u++)
#pragma unroll
          for (int k = 0; k < kComp; k++) x[u][k] = xp[16 * (i0 + u) * kXWords<TX> + k];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < UD; u++)
#pragma unroll
          for (int j = 0; j < 4; j++)
#pragma unroll
            for (int k = 0; k < kComp; k++) f[j][k] += q[u][j >> 1][j & 1] * x[u][k];
      };
      load(0, ca);
      for (int i0 = 0; i0 < ni; i0 += 2 * UD) {
        load(min(i0 + UD, ni - UD), cb);
        __builtin_amdgcn_sched_barrier(0);
        mac(i0, ca);
        __builtin_amdgcn_sched_barrier(0);
        if (i0 + UD >= ni) break;
        load(min(i0 + 2 * UD, ni - UD), ca);
        __builtin_amdgcn_sched_barrier(0);
        mac(i0 + UD, cb);
        __builtin_amdgcn_sched_barrier(0);
      }
      // sum over the sixteen slices: the wave's halves, then its rows of 16 lanes,
      // exchange orbitals (half h ends with orbitals 2h, 2h + 1, row parity
      // with one of them), then the slices of a row
      double e[kComp];
#pragma unroll
      for (int k = 0; k < kComp; k++) {
        const double h0 = swap32_add(f[0][k], f[2][k]), h1 = swap32_add(f[1][k], f[3][k]);
        double x = swap16_add(h0, h1);
        x += dpp_f64<0x124>(x);  // row_ror:4, row_ror:8
        x += dpp_f64<0x128>(x);
        e[k] = x;
      }
      const int o = (lane & 32 ? NC / 2 : 0) + g2_ + ((lane >> 4) & 1);
      if ((lane & 12) == 0 && o < n)
#pragma unroll
        for (int k = 0; k < kComp; k++) s_v[k][o] = e[k];
    }
    if (A.has_cusp) {
      // electron-nucleus cusp replacement of the row (cusp.hip), one thread
      // per orbital (NT >= n) over the nuclei within their largest radius
      __syncthreads();
      const CuspDev &cu = A.cusp[sp];
      double e5[kComp] = {0, 0, 0, 0, 0};
      bool hit = false;
      for (int a0 = 0; a0 < nn; a0 += 64) {
        bool near = false;
        if (a0 + lane < nn) {
          const double rcm = cu.rc_max[a0 + lane];
          const double *at = s_nuc + 4 * (a0 + lane);
          const double dx = xn[0] - at[0], dy = xn[1] - at[1], dz = xn[2] - at[2];
          near = dx * dx + dy * dy + dz * dz < rcm * rcm;
        }
        unsigned long long hits = __ballot(near);
        while (hits) {
          const int a_ = a0 + __builtin_ctzll(hits);
          hits &= hits - 1;
          const double dx = xn[0] - s_nuc[4 * a_], dy = xn[1] - s_nuc[4 * a_ + 1],
                       dz = xn[2] - s_nuc[4 * a_ + 2];
          const double r2 = dx * dx + dy * dy + dz * dz, rr = sqrt(r2);
          if (t >= n) continue;
          const double *f = cu.orb8 + ((long)a_ * cu.norb + t) * 8;
          if (!(rr < f[0])) continue;
          hit = true;
          // original s-type part on this nucleus
          const double *cf = cu.s_coef + (long)t * cu.ns;
          for (int g = cu.s_off[a_]; g < cu.s_off[a_ + 1]; g++) {
            const double a0_ = cu.s_alpha[g];
            const double te = cf[g] * exp(-a0_ * r2);
            const double tg = -2 * a0_ * te;
            e5[0] -= te;
            e5[1] -= dx * tg;
            e5[2] -= dy * tg;
            e5[3] -= dz * tg;
            e5[4] -= 2 * a0_ * (2 * a0_ * r2 - 3) * te;
          }
          // replacement C + sgn0 exp(alpha(r))
          double pf = f[7], pd = 0.0, pd2 = 0.0;
          for (int i = 3; i >= 0; i--) {
            pd2 = pd2 * rr + pd;
            pd = pd * rr + pf;
            pf = pf * rr + f[3 + i];
          }
          pd2 *= 2;
          const double e = f[2] * exp(pf);
          const double tg = e * pd / rr;
          e5[0] += f[1] + e;
          e5[1] += tg * dx;
          e5[2] += tg * dy;
          e5[3] += tg * dz;
          e5[4] += e * (pd2 + pd * (2.0 / rr + pd));
        }
      }
      if (hit)
#pragma unroll
        for (int k = 0; k < kComp; k++) s_v[k][t] = (double)(TX)(s_v[k][t] + e5[k]);
    }
    __syncthreads();
    // ---- w(c) = v A^-1(:, c), the sums T1 and T2, and the moved electron's own
    double wc = 0.0, T1[NK], T2[NK];
    {
      double p1[KC], p2[KC];
#pragma unroll
      for (int k = 0; k < KC; k++) p1[k] = p2[k] = 0.0;
      const double *v0 = s_v[0] + o_beg, *co = col + sl * RI;
#pragma unroll
      for (int i0 = 0; i0 < RI; i0 += U8) {
        if (i0 < rows) {  // a, d and col are zero past the slice
          double v8[U8], c8[U8];
#pragma unroll
          for (int i = 0; i < U8; i++) {
            v8[i] = v0[i0 + i];
            if constexpr (RD) c8[i] = co[i0 + i];
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < U8; i++) {
            wc += v8[i] * a[i0 + i];
            if constexpr (RD) {
#pragma unroll
              for (int k = 0; k < KC; k++) {
                p1[k] += (double)d[i0 + i][k] * a[i0 + i];
                p2[k] += (double)d[i0 + i][k] * c8[i];
              }
            }
          }
        }
      }
      if constexpr (SL == 2) {
        wc += dpp_f64<0xB1>(wc);
#pragma unroll
        for (int j = 0; j < NK; j++) {
          constexpr int J2 = ONE ? 0 : NK;
          const double k1 = sl ? p1[J2 + j] : p1[j], s1 = sl ? p1[j] : p1[J2 + j];
          const double k2 = sl ? p2[J2 + j] : p2[j], s2 = sl ? p2[j] : p2[J2 + j];
          T1[j] = k1 + dpp_f64<0xB1>(s1);
          T2[j] = k2 + dpp_f64<0xB1>(s2);
        }
      } else if constexpr (F32) {
        wc = quad_ordered(wc);
        T1[0] = quad_ordered_own(p1[0], p1[1], p1[2], p1[3], sl);
        T2[0] = quad_ordered_own(p2[0], p2[1], p2[2], p2[3], sl);
      } else {
        wc = quad_sum(wc);
        if constexpr (RD) {
          T1[0] = quad_sum_own(p1[0], p1[1], p1[2], p1[3], sl);
          T2[0] = quad_sum_own(p2[0], p2[1], p2[2], p2[3], sl);
        } else {
          T1[0] = t1;
          T2[0] = myacc >= 0 ? s_fix[max(myacc, 0)][sl] : G[0];
        }
      }
      if (sl == 0 && c < n && grp == 0) s_wv[c] = wc;
    }
    if (wave == 0 || (NARROW && wave == 1)) {
      const bool held = NARROW && wave == 1;
      double f[4] = {0, 0, 0, 0};
#pragma unroll
      for (int h = 0; h < (NC + 63) / 64; h++)
        if (lane + 64 * h < n)
#pragma unroll
          for (int k = 0; k < 4; k++) {
            const double x = s_v[1 + k][lane + 64 * h];
            f[k] += (held ? (double)(TS)x : as_stored<TS>(x)) * col[cl[h]];
          }
#pragma unroll
      for (int k = 0; k < 4; k++) f[k] = wave_sum(f[k]);
      if (lane == 0)
#pragma unroll
        for (int k = 0; k < 4; k++) (held ? s_held : s_new)[k] = f[k];
    }
    __syncthreads();
    const double ratio = s_wv[r];
    const bool rok = (ratio != 0.0) && isfinite(ratio);
    const double qinv = 1.0 / ratio;
    double gown[NK];
#pragma unroll
    for (int j = 0; j < NK; j++) {
      const int k = grp * KC + (ONE ? 0 : sl * NK) + j;
      gown[j] = c == r ? s_new[k] * qinv : T1[j] - wc * qinv * T2[j];
      if (c < n) s_gq[k][c] = gown[j];
    }
    __syncthreads();
    auto jsum = [&](int k) {
      double x = 0.0;
#pragma unroll
      for (int i = 0; i < NW; i++) x += s_wj[k][i];
      return x;
    };
    // ---- gradients and Green's function sums (QMCWalker.cpp:343-398, 756-780)
    // over all electrons, thread e electron e
    double gnew[3] = {0, 0, 0}, ft = 1.0;
    int ct = cn;
    if (qf && wave == m >> 6) {
      // nearest nucleus of the proposal (first of equals)
      double best = 1e300;
      int bi = 0;
      for (int a0 = 0; a0 < nn; a0 += 64) {
        const double rr = a0 + lane < nn ? s_rn[a0 + lane] : 1e300;
        const double mn = wave_min(rr);
        if (mn < best) {
          best = mn;
          bi = a0 + __builtin_ctzll(__ballot(rr == mn));
        }
      }
      if (t == m) ct = bi;
    }
    double lsum = 0, fwd = 0, rev = 0, lapc = 0, gsq = 0, vbt = 0, vbo = 0, vo = 0;
    if (t < N) {
      const bool same = esp == sp;
      if (same) lapc = s_gq[3][ee_];
      if (t == m)
#pragma unroll
        for (int k = 0; k < 3; k++) un_[k] = jsum(4 + k);
      double g[3], gc[3];
#pragma unroll
      for (int k = 0; k < 3; k++) {
        gnew[k] = same ? s_gq[k][ee_] : ge[k];
        const double ux = un_[k];
        g[k] = gnew[k] + ux;
        gc[k] = ge[k] + Ue[k];
        lsum += ux * gnew[k] * 2.0;
        lsum += ux * ux;
        gsq += g[k] * g[k];
      }
      if (qf) {
        const double x[3] = {t == m ? xn[0] : Re[0], t == m ? xn[1] : Re[1], t == m ? xn[2] : Re[2]};
        ft = drift_factor_lds(g, x, s_nuc + 4 * ct, tau);
        double g2 = 0.0, gc2 = 0.0;
#pragma unroll
        for (int k = 0; k < 3; k++) { g2 += g[k] * g[k]; gc2 += gc[k] * gc[k]; }
        vbt = ft * ft * g2;
        vbo = fo * fo * gc2;
        vo = gc2;
      }
#pragma unroll
      for (int k = 0; k < 3; k++) {
        if (t != m) {
          fwd += tau * fo * gc[k] * tau * fo * gc[k];
          rev += tau * ft * g[k] * tau * ft * g[k];
        } else {
          const double tt = Re[k] - xn[k] - tau * ft * g[k], chi = sqt * draw[k];
          rev += tt * tt;
          fwd += chi * chi;
        }
      }
    }
    {
      double vals[8] = {lsum, fwd, rev, lapc, gsq, vbt, vbo, vo};
#pragma unroll
      for (int k = 0; k < 8; k++) {
        if (k >= 5 && !qf) break;
        const double sm = wave_sum(vals[k]);
        if (lane == 0) s_red[k][wave] = sm;
      }
    }
    __syncthreads();
    // ---- Metropolis with the Green's function ratio (QMCWalker.cpp:1578-1685),
    // the same in every thread
    auto rsum = [&](int k) {
      double x = 0.0;
#pragma unroll
      for (int i = 0; i < NW; i++) x += s_red[k][i];
      return x;
    };
    gsq = rsum(4);
    const bool sing = sing0 || !rok || !(gsq > 0.0) || !isfinite(gsq);
    const double lratio = log(fabs(ratio)), U_old = s_psi[pb][0];
    const double ld_s = s_psi[pb][1 + sp], ld_o = s_psi[pb][2 - sp], U = U_old + jsum(0);
    const double logpsi_new = ld_s + lratio + ld_o + U, logpsi_old = ld_s + ld_o + U_old;
    double p = sing ? 0.0
                    : exp(2.0 * (logpsi_new - logpsi_old) - (rsum(2) - rsum(1)) / (2.0 * tau));
    if (!(p == p)) p = 0.0;
    else if (!sing) p = old_walker_boost(p, age, A.walk.old_walker);
    if (A.mode == 2 && ratio < 0) p = 0.0;
    if (p > 1.0) p = 1.0;
    const bool accept = p > draw[3];
    age = accept ? 0 : age + 1;  // QMCWalker.cpp:1656-1672
    if (t == 0) {
      const double lap_s = rsum(3);
      const double Uxx = s_sc[1] + jsum(1), Vee = s_sc[2] + jsum(2), Ven = s_sc[3] + jsum(3);
      const double lapR = lap_s + s_sc[10 - sp] + Uxx + rsum(0);
      const double V = A.v_nn + Vee + Ven;
      const double EL = -0.5 * lapR + V;
      const double el_old = s_sc[4], el = accept ? EL : el_old;
      double wt = 1.0;
      if (A.mode == 2) {
        // umrigar93_probability_weighted reweighting once per electron sweep
        // (QMCWalker.cpp:1060-1185, UNR93 eq. 25, 33-34)
        wt = s_sc[11];
        if (A.reweight && m == 0) {
          double so_, st_;
          if (A.energy_mod) {
            const double mr_t = (qf && gsq > 0.0) ? sqrt(rsum(5)) / sqrt(gsq) : 1.0;
            const double vo_ = qf ? rsum(7) : 0.0;
            const double mr_o = (qf && vo_ > 0.0) ? sqrt(rsum(6)) / sqrt(vo_) : 1.0;
            so_ = (A.e_trial - A.e_est) + (A.e_est - el_old) * mr_o;
            st_ = (A.e_trial - A.e_est) + (A.e_est - EL) * mr_t;
          } else {
            so_ = A.e_trial - el_old;
            st_ = A.e_trial - EL;
          }
          if (!(p > 0.0)) st_ = 0.0;
          const double dW = exp(A.tau_eff * (p * 0.5 * (so_ + st_) + (1.0 - p) * so_));
          wt = reweight_walker(wt, dW, age, el, A.walk);
          s_sc[11] = wt;
        }
        s_sc[16] += wt;
      }
      s_sc[12] += wt * el;
      s_sc[13] += wt * el * el;
      s_sc[14] += accept ? 1.0 : 0.0;
      s_sc[15] += sing ? 0.0 : EL;
      if (m == 0 && A.obs) {
        // estimator p E_L(R') + (1 - p) E_L(R) (QMCWalker.cpp:2096-2104)
        double *ob = A.obs + 3 * ((long)obs_row * A.obs_stride + b);
        ob[0] = p > 0.0 ? p * EL + (1.0 - p) * el_old : el_old;
        ob[1] = wt;
        ob[2] = p;
      }
      if (accept) {
        s_sc[0] = U; s_sc[1] = Uxx; s_sc[2] = Vee; s_sc[3] = Ven; s_sc[4] = EL;
        s_sc[5 + sp] = ld_s + lratio;
        if (ratio < 0) s_sc[7 + sp] = -s_sc[7 + sp];
        s_sc[9 + sp] = lap_s;
      }
      // the next step's copy (this one is still being read by other waves)
      s_psi[pb ^ 1][0] = s_sc[0];
      s_psi[pb ^ 1][1] = s_sc[5];
      s_psi[pb ^ 1][2] = s_sc[6];
    }
    if (m == 0) obs_row++;
    if (accept) {
      // A'^-1 = A^-1 - A^-1(:, r) z^T, z(c) = (w(c) - delta_cr) / ratio
      const double z = (wc - (c == r ? 1.0 : 0.0)) * qinv;
#pragma unroll
      for (int i0 = 0; i0 < RI; i0 += U8) {
        if (i0 < rows) {
          double c8[U8];
#pragma unroll
          for (int i = 0; i < U8; i++) c8[i] = col[sl * RI + i0 + i];
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < U8; i++) a[i0 + i] -= c8[i] * z;
        }
      }
      if constexpr (!RD) {
        t1 = NARROW && c == r ? s_held[sl] * qinv : gown[0];
        if (c == r) myacc = nacc;
      }
      fo = ft;
      cn = ct;
#pragma unroll
      for (int k = 0; k < 3; k++) {
        Ue[k] = un_[k];
        ge[k] = gnew[k];
        if (t == m) Re[k] = xn[k];
      }
      // the moved electron's column of the value and derivative matrices
      TS *dmw = (TS *)A.s[sp].dmat + (long)w * kDer * n * n;
      double *dvw = A.s[sp].dval + (long)w * n * n;
      for (int o = t; o < n; o += NT) {
        const double v4[4] = {s_v[1][o], s_v[2][o], s_v[3][o], s_v[4][o]};
        dvw[(long)o * n + r] = s_v[0][o];
        st_der(dmw + 4 * ((long)o * n + r), v4[0], v4[1], v4[2], v4[3]);
        if constexpr (!RD)
#pragma unroll
          for (int k = 0; k < 4; k++) s_vrow[(nacc * NC + o) * 4 + k] = (double)(TS)v4[k];
      }
      if constexpr (RD) {
        if (c == r) {
#pragma unroll
          for (int i = 0; i < RI; i++) {
            const double in = i < rows && o_beg + i < n ? 1.0 : 0.0;  // o_beg + i < NC always
#pragma unroll
            for (int k = 0; k < KC; k++)
              d[i][k] = (TD)(in * as_stored<TS>(s_v[1 + KC * grp + k][o_beg + i]));
          }
        }
      }
    }
    if constexpr (!RD) {
      // T2 of the block's remaining columns: A'^-1(:, r + j) = A^-1(:, r + j) - A^-1(:, r) z(r + j)
#pragma unroll
      for (int j = 1; j < KB; j++) {
        const double z = (accept && r + j < n) ? s_wv[r + j] * qinv : 0.0;
        G[j - 1] = G[j] - z * T2[0];
      }
      if (accept) nacc++;
      blk_left--;
    }
  }
  }
  // ---- state out
  store_inv(cur);
  if constexpr (!RD) {
    const int left = A.keep ? blk_left : 0, n4 = 4 * n;
    if (left > 0) {
      double *cb = A.carry + (long)w * (8 * KB * nu);
      __syncthreads();  // the last move's row in s_vrow
      if (t < n4) {
        cb[t] = t1;
        cb[n4 + t] = myacc;
        for (int i = 0; i < nacc; i++) cb[(2 + i) * n4 + t] = s_vrow[i * NT + t];
#pragma unroll
        for (int j = 0; j < KB - 1; j++) cb[(1 + KB + j) * n4 + t] = G[j];
      }
    }
    if (t == 0) A.s[cur].carried[w] = left > 0 ? left | nacc << 4 | (m_next + 1) << 8 : 0;
  }
  if (t < N) {
    const long e = (long)w * N + t;
    double *gp = A.s[esp].gradPR + ((long)w * (esp ? N - nu : nu) + ee_) * 3;
    for (int k = 0; k < 3; k++) {
      A.R[3 * e + k] = Re[k];
      A.Ux[3 * e + k] = Ue[k];
      gp[k] = ge[k];
    }
  }
  if (t == 0) {
    A.U[w] = s_sc[0]; A.Uxx[w] = s_sc[1]; A.Vee[w] = s_sc[2]; A.Ven[w] = s_sc[3];
    A.cur_el[w] = s_sc[4];
    for (int s = 0; s < 2; s++)
      if (s == 0 || N > nu) {
        A.s[s].logdet[w] = s_sc[5 + s];
        A.s[s].sgn[w] = s_sc[7 + s];
        A.s[s].lapPR[w] = s_sc[9 + s];
      }
    if (A.walk.age) A.walk.age[w] = age;
    A.acc_el[w] = s_sc[12]; A.acc_el2[w] = s_sc[13]; A.acc_n[w] = s_sc[14];
    A.acc_prop_el[w] = s_sc[15];
    if (A.mode == 2) {
      A.weight[w] = s_sc[11];
      A.acc_w[w] = s_sc[16];
    }
  }
}

namespace {

// dynamic LDS of the launch: basis values, tables and scratch (walk_kernel's
// layout; the last term of the sum is more than its rounding to even lengths)
size_t walk_lds(int NC, int B, int kpad, int nn, int nshell, int np, int mn, int md, size_t tx) {
  const size_t ps = 1 + mn + md;
  size_t d = 3 * (size_t)np + 5 * (size_t)nn + (3 + 2 * (size_t)nn) * ps + (size_t)B;
  if (tx == 8 && NC > 32) d += 5 * (size_t)NC * walk_block(NC);
  return (size_t)kpad * (tx == 4 ? 8 : 5) * tx + 8 * d + 4 * ((size_t)np + nshell + 1);
}

constexpr size_t kLdsBytes = 160 * 1024;
// the kernel's static LDS, an upper bound over the tiles
size_t walk_static_lds(int NC) {
  return 8 * (size_t)(2 * NC + kComp * NC + NC + 4 * NC + 15 * 8 + 64 * 4 + 12 + 8 + 4 * 8 + 23) +
         256;
}

}  // namespace

bool walk_fits(int n_up, int n_dn, int B, int kpad, int nn, int nshell, int np, int mn, int md, size_t tx) {
  if (n_up < 1 || n_up > 128 || (tx != 8 && tx != 4)) return false;
  // FP32 operands beyond 64 electrons a spin: the columns of A^-1 and the
  // derivative matrices, in the two slices the bits ask for, are more than a
  // CU's registers hold without spilling (200 electrons, 512 walkers: 2.5 ms
  // for 16 steps in two rounds of 256, 2.9 ms step by step; 8192 walkers of
  // 256 electrons: 1.7 against 0.93 ms a step)
  if (tx == 4 && n_up > 64) return false;
  // Beyond 32 electrons a spin the batch decides between this kernel and the
  // steps, which then have to give a walker the same bits: they do with the same
  // slices of a column, two but in the steps' 16-column tile, which has four
  if (tx == 4 && n_up > 32 && n_dn > 0 && n_dn <= 16) return false;
  if (np >= 1 << 16 || nn >= 1 << 20 || kpad % (tx == 4 ? 48 : 32)) return false;  // packed function records
  const int NC = walk_tile(n_up);
  return walk_lds(NC, B, kpad, nn, nshell, np, mn, md, tx) + walk_static_lds(NC) <= kLdsBytes;
}

long walk_carry_len(int n_up, size_t tx) {
  return tx == 8 && n_up > 32 ? 8L * walk_block(walk_tile(n_up)) * n_up : 0;
}

template <typename TS, typename TX, int NC>
static hipError_t launch_tile(const WalkArgs &a, const int *walkers, int num, hipStream_t st) {
  const size_t lds = walk_lds(NC, a.B, a.kpad, a.nn, a.nshell, a.np, a.pade_mn, a.pade_md,
                              sizeof(TX));
  auto k = walk_kernel<TS, TX, NC>;
  if (lds > 48 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k, dim3(num), dim3(walk_threads<TX, NC>()), lds, st, a, walkers, num);
  return hipGetLastError();
}

template <typename TS, typename TX>
hipError_t launch_walk(const WalkArgs &a, const int *walkers, int num, hipStream_t st) {
  if (num <= 0 || a.nsteps <= 0) return hipSuccess;
  if (!walk_fits(a.n_up, a.N - a.n_up, a.B, a.kpad, a.nn, a.nshell, a.np, a.pade_mn, a.pade_md,
                 sizeof(TX)) ||
      !a.tab || a.tab_len % 2 != 0 ||
      a.tab_len < walk_tab_len(a.B, a.nn, a.np, a.pade_mn, a.pade_md) ||
      a.N > 2 * a.n_up || (walk_carry_len(a.n_up, sizeof(TX)) > 0 && (!a.carry || !a.s[0].carried)))
    return hipErrorInvalidValue;
  const int NC = walk_tile(a.n_up);
  if (NC == 16) return launch_tile<TS, TX, 16>(a, walkers, num, st);
  if (NC == 32) return launch_tile<TS, TX, 32>(a, walkers, num, st);
  if (NC == 64) return launch_tile<TS, TX, 64>(a, walkers, num, st);
  if constexpr (sizeof(TX) == 8) {
    if (NC == 96) return launch_tile<TS, TX, 96>(a, walkers, num, st);
    return launch_tile<TS, TX, 128>(a, walkers, num, st);
  }
  return hipErrorInvalidValue;
}

template hipError_t launch_walk<double, double>(const WalkArgs &, const int *, int, hipStream_t);
template hipError_t launch_walk<float, float>(const WalkArgs &, const int *, int, hipStream_t);
template hipError_t launch_walk<float, double>(const WalkArgs &, const int *, int, hipStream_t);
template hipError_t launch_walk<bf16s, float>(const WalkArgs &, const int *, int, hipStream_t);

}  // namespace qmcb
