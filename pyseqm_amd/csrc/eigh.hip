// FP64 density step by diagonalisation, one workgroup per molecule (blocks up to 192 orbitals):
// P = 2 C_occ C_occ^T of the packed Fock block (sym_eig_trunc, seqm/seqm_functions/diag.py:110-241,
// as the SCF's make_Pnew uses it, scf_loop.py:55-103), without padding the block to a batch size.
//
//   1. Householder reduction of the block to tridiagonal form T = Q^T F Q (dsytd2 order), with the
//      matrix in registers (tridiagonalise below).  The reflectors go to the global workspace.
//   2. The nocc lowest eigenvalues of T by Sturm counts: one evenly spaced grid over the whole
//      spectrum for all of them, then multisection (a group of lanes per eigenvalue) to 1e-11 |T|,
//      closer where a neighbour is within 1e-6 |T|, to rounding within 1e-9 |T|.
//   3. Their eigenvectors from twisted factorisations of T - lambda I, two lanes per vector (one from
//      each end), the vectors in LDS: one factorisation at the bracket's middle, whose Rayleigh
//      correction is kept unrounded beside lambda, and one there.
//   4. Vectors of eigenvalues closer than 1e-3 |T| (a cluster) orthogonalised against each other,
//      a cluster per wave.  Vectors further apart come out orthogonal to eps |T| / gap.  Where a
//      neighbour is closer than 1e-10 |T| (a degenerate level, which a twisted factorisation would
//      give the same vector twice) the vectors come from inverse iteration with different starts
//      instead, orthogonalised between its solves: they span the level's subspace (P depends on the
//      occupied subspace only).
//   5. Back-transformation C = Q Z by blocks of 16 reflectors and P = 2 C C^T, both on FP64 MFMA
//      tiles.
// Every reduction runs in a fixed order: reruns are bitwise identical.
#include "common.h"

using namespace pyseqm;

typedef double doublex4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int kEighMaxN = 192;      // largest block this solver takes
constexpr int kLdsDoubles = 20480;  // 160 KiB of LDS
constexpr int kLdsFixed = 32;       // of them the kernel's own 256 bytes (__syncthreads_or)
constexpr int kLdsLaunch = kLdsDoubles - kLdsFixed;  // what a launch can ask for
constexpr int kTPanel = 256;        // doubles of one panel's 16 x 16 T factor
constexpr int kLdsExtra = 25;       // doubles of the twist rows and of an alignment gap

// workspace per listed molecule, in doubles, at slot * 4 * nmax^2:
//   [0, nmax^2)          reflectors: row i holds u_i (zero at columns <= i of its panel of 16)
//   [nmax^2, 4 nmax^2)   element k of vector j at k * nmax + j: the lower multipliers of the twisted
//                        factorisations (blocks above 48 orbitals), the U factor of each
//                        inverse-iteration LU (reciprocal diagonal and two superdiagonals); then
//                        the panels' T factors of the back-transformation (above 48 orbitals)
// LDS: eigenvectors n x ldz (before them, in the same place, the Householder vectors, then the grid's
// counts), (d, e^2) pairs, e, eigenvalues, reflector scales and vector scales (n each), the twist
// rows (a byte each), and for blocks of up to 48 orbitals the panels' T factors and the lower
// multipliers.  The variant follows the launch's largest block nmax.
__host__ __device__ inline int grid_slots(int nmax) { return nmax <= 48 ? 48 : (nmax <= 96 ? 96 : 192); }
// The size rule of the entry points: n nocc + 3 n + 3 S + 128 doubles (S: the variant's 48 / 96 /
// 192 grid rows) of the 20480.  lds_doubles, what a launch asks for, stays within kLdsLaunch for every
// accepted block: with the even stride it is n nocc + 6 n + 25 <= 20480 + 3 n - 679 <= 20377.
__host__ __device__ inline int rule_doubles(int n, int nv) { return n * nv + 3 * n + 3 * grid_slots(n) + 128; }
// Row stride of the eigenvectors: odd where that fits (rows of 16 lanes then fall on distinct LDS
// banks), else nv.
__host__ __device__ inline int zstride(int n, int nv) {
  return n * (nv | 1) + 6 * n + kLdsExtra <= kLdsLaunch ? (nv | 1) : nv;
}
// Doubles of the eigenvector region: also holds the Householder vectors (2 S) and the grid's counts
// (two ints per thread) before.
__host__ __device__ inline int zregion(int n, int nv, int S) {
  const int z = n * zstride(n, nv), least = S == 192 ? 512 : (S == 96 ? 256 : 96);
  return z > least ? z : least;
}
inline int lds_doubles(int nmax, int nv) {
  const int S = grid_slots(nmax);
  // where the odd stride does not fit the largest block it may still fit a smaller one of the launch
  if (zstride(nmax, nv) != (nv | 1)) return kLdsLaunch;
  return zregion(nmax, nv, S) + 6 * nmax + kLdsExtra + (S == 48 ? 3 * kTPanel + nmax * (nv | 1) : 0);
}

template <int NT>
__device__ inline double eig_block_max(double v, double* red) {
  constexpr int NW = NT / 64;
  for (int o = 1; o < 64; o <<= 1) v = fmax(v, __shfl_xor(v, o));
  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __syncthreads();
  if (lane == 0) red[wid] = v;
  __syncthreads();
  double s = red[0];
#pragma unroll
  for (int k = 1; k < NW; ++k) s = fmax(s, red[k]);
  return s;
}

template <int NT>
__device__ inline double eig_block_min(double v, double* red) {
  constexpr int NW = NT / 64;
  for (int o = 1; o < 64; o <<= 1) v = fmin(v, __shfl_xor(v, o));
  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __syncthreads();
  if (lane == 0) red[wid] = v;
  __syncthreads();
  double s = red[0];
#pragma unroll
  for (int k = 1; k < NW; ++k) s = fmin(s, red[k]);
  return s;
}

// 1 / q to full FP64 accuracy without the scaled division sequence: v_rcp_f64 and two Newton
// steps (q is kept away from zero and overflow by the caller's pivmin)
__device__ inline double rcp_f64(double q) {
  double r = __builtin_amdgcn_rcp(q);
  r = fma(fma(-q, r, 1.0), r, r);
  r = fma(fma(-q, r, 1.0), r, r);
  return r;
}

// cnt[i] = number of eigenvalues of the tridiagonal de[k] = (d_k, e_k^2) below x[i]: the negative
// pivots q_k of the LDL^T factorisation of T - x I, counted as sign changes of the Sturm sequence
// p_0 = 1, p_k = (d_k - x) p_{k-1} - e2_{k-1} p_{k-2} (q_k = p_k / p_{k-1}), whose dependent chain
// is one FMA per step instead of a reciprocal.  Every e2 is above zero (the caller floors it at
// (1e-30 |T|)^2), so a p_k of exactly zero is followed by one of the sign opposite to p_{k-1}: one
// sign change over the two steps whichever sign bit the zero carries.  Signs collect in the bits of
// one register (one instruction a step); every 8 steps they are counted and both terms scaled
// by the same power of two (exact; signs and ratios unchanged), which keeps them in range.
template <int K>
__device__ inline void sturm_counts(const double2* de, int n, const double (&x)[K], int (&cnt)[K]) {
  double p0[K], p1[K];
  unsigned m[K];
#pragma unroll
  for (int i = 0; i < K; ++i) {
    p0[i] = 1.0;
    p1[i] = de[0].x - x[i];
    m[i] = (unsigned)__double2hiint(p1[i]) >> 31;
    cnt[i] = (int)m[i];
  }
  auto step = [&](double dk, double e2k) {
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const double p2 = fma(dk - x[i], p1[i], -(e2k * p0[i]));
      m[i] = __builtin_amdgcn_alignbit(m[i], (unsigned)__double2hiint(p2), 31);  // m << 1 | sign
      p0[i] = p1[i];
      p1[i] = p2;
    }
  };
  // the next eight rows are read while eight are used (reads past row n - 1 fall into the arrays
  // that follow de and are not used)
  int k = 1;
  double prev = de[0].y;
  double2 w[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) w[t] = de[1 + t];
#pragma unroll 2
  for (; k + 8 <= n; k += 8) {
    double2 wn[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) wn[t] = de[k + 8 + t];
    step(w[0].x, prev);
#pragma unroll
    for (int t = 1; t < 8; ++t) step(w[t].x, w[t - 1].y);
    prev = w[7].y;
#pragma unroll
    for (int t = 0; t < 8; ++t) w[t] = wn[t];
#pragma unroll
    for (int i = 0; i < K; ++i) {
      cnt[i] += __popc((m[i] ^ (m[i] >> 1)) & 0xffu);
      const int ex = max(__builtin_amdgcn_frexp_exp(p0[i]), __builtin_amdgcn_frexp_exp(p1[i]));
      p0[i] = __builtin_amdgcn_ldexp(p0[i], -ex);
      p1[i] = __builtin_amdgcn_ldexp(p1[i], -ex);
    }
  }
  const unsigned rest = (1u << (n - k)) - 1u;
#pragma unroll
  for (int t = 0; t < 7; ++t)
    if (k + t < n) step(w[t].x, t == 0 ? prev : w[t > 0 ? t - 1 : 0].y);
#pragma unroll
  for (int i = 0; i < K; ++i) cnt[i] += __popc((m[i] ^ (m[i] >> 1)) & rest);
}

// One DPP lane permutation of a double (two 32-bit DPP moves; VALU, no LDS round trip).
// Every control used here (quad permutations, row mirrors) names a source lane inside the row for
// every lane, so no lane keeps an old value and none needs initialising.
template <int CTRL>
__device__ inline double dpp_f64(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Sum / max / min over aligned groups of t lanes (t a power of two, the same in every lane):
// DPP within a 16-lane row, shuffles across rows.
__device__ inline double group_sum_t(double v, int t) {
  if (t >= 2) v += dpp_f64<0xB1>(v);
  if (t >= 4) v += dpp_f64<0x4E>(v);
  if (t >= 8) v += dpp_f64<0x141>(v);
  if (t >= 16) v += dpp_f64<0x140>(v);
  if (t >= 32) v += __shfl_xor(v, 16);
  if (t >= 64) v += __shfl_xor(v, 32);
  return v;
}
__device__ inline double group_max_t(double v, int t) {
  if (t >= 2) v = fmax(v, dpp_f64<0xB1>(v));
  if (t >= 4) v = fmax(v, dpp_f64<0x4E>(v));
  if (t >= 8) v = fmax(v, dpp_f64<0x141>(v));
  if (t >= 16) v = fmax(v, dpp_f64<0x140>(v));
  if (t >= 32) v = fmax(v, __shfl_xor(v, 16));
  if (t >= 64) v = fmax(v, __shfl_xor(v, 32));
  return v;
}
__device__ inline double group_min_t(double v, int t) {
  if (t >= 2) v = fmin(v, dpp_f64<0xB1>(v));
  if (t >= 4) v = fmin(v, dpp_f64<0x4E>(v));
  if (t >= 8) v = fmin(v, dpp_f64<0x141>(v));
  if (t >= 16) v = fmin(v, dpp_f64<0x140>(v));
  if (t >= 32) v = fmin(v, __shfl_xor(v, 16));
  if (t >= 64) v = fmin(v, __shfl_xor(v, 32));
  return v;
}

// deterministic pseudo-random start vector element in (-1, 1)
__device__ inline double start_value(int j, int k) {
  unsigned h = (unsigned)j * 2654435761u + (unsigned)k * 40503u + 12345u;
  h ^= h >> 15;
  h *= 2246822519u;
  h ^= h >> 13;
  return (double)h * (2.0 / 4294967296.0) - 1.0;
}


// One end's multipliers L_k = e_k / q_k of T - (hi + lo) I for the vector of this lane, q_k = p_k /
// p_{k-1} with p_k the Sturm sequence from that end (DIR 1: from the top, -1: from the bottom), so
// that the chain has no division.  out walks by os per row.  A p_k of zero is floored at tiny
// p_{k-1}.  d and e point at this end's first entries; rows are read eight ahead of their use (at
// most eight past the other end, into the LDS arrays around; not used there).
template <int DIR, class P>
__device__ __forceinline__ void twisted_sweep(const double2* d, const double* e, int n, double hi, double lo,
                                              double tiny, P out, int os) {
  double p0 = 1.0, p1 = (d[0].x - hi) - lo;
  if (fabs(p1) < tiny) p1 = tiny;
  auto step = [&](double dk, double ek) {
    const double ep0 = ek * p0;
    *out = ep0 * rcp_f64(p1);
    out += os;
    double p2 = fma((dk - hi) - lo, p1, -(ek * ep0));
    const double f = tiny * p1;
    p2 = fabs(p2) < fabs(f) ? f : p2;
    p0 = p1;
    p1 = p2;
  };
  double w[8], x[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    w[t] = d[DIR * (t + 1)].x;
    x[t] = e[DIR * t];
  }
  int k = 0;
#pragma unroll 2
  for (; k + 8 < n; k += 8) {
    double wn[8], xn[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      wn[t] = d[DIR * (k + 9 + t)].x;
      xn[t] = e[DIR * (k + 8 + t)];
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) step(w[t], x[t]);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      w[t] = wn[t];
      x[t] = xn[t];
    }
    const int ex = max(__builtin_amdgcn_frexp_exp(p0), __builtin_amdgcn_frexp_exp(p1));
    p0 = __builtin_amdgcn_ldexp(p0, -ex);
    p1 = __builtin_amdgcn_ldexp(p1, -ex);
  }
#pragma unroll
  for (int t = 0; t < 8; ++t)
    if (k + t + 1 < n) step(w[t], x[t]);
}

// One step of inverse iteration on T - sig I, one thread, from a fixed pseudo-random start (of vector j) or from
// z as it is; z (stride ldz) ends scaled to a largest element of 1.  Returns 1 / |z|.
__device__ __forceinline__ double inverse_iteration(const double2* de, const double* e, double* z, int ldz, double* U0,
                                                    double* U1, double* U2, int ldu, int n, int j, double sig,
                                                    double tiny, bool start) {
  if (start)
    for (int k = 0; k < n; ++k) z[k * ldz] = start_value(j, k);
  // LU of T - sig I with partial pivoting, the right-hand side eliminated alongside; the
  // running row and right-hand side stay in registers, U goes to the workspace.  Each step
  // keeps one of two rows as the pivot row (its diagonal and sub-diagonal entries compared)
  // and eliminates the other, both cases as one select-based update (lanes differ in their
  // choices); the next step's d, e and right-hand side are read from LDS one step ahead.
  double diag = de[0].x - sig, sup = n > 1 ? e[0] : 0.0;
  double yk = z[0];
  double sub_n = n > 1 ? e[0] : 0.0, dn_n = n > 1 ? de[1].x : 0.0, ns_n = n > 2 ? e[1] : 0.0;
  double y_n = n > 1 ? z[ldz] : 0.0;
  for (int k = 0; k + 1 < n; ++k) {
    const double sub = sub_n, nd = dn_n - sig, ns = ns_n, yk1 = y_n;
    if (k + 2 < n) {
      sub_n = ns_n;
      dn_n = de[k + 2].x;
      ns_n = k + 3 < n ? e[k + 2] : 0.0;
      y_n = z[(k + 2) * ldz];
    }
    const size_t o = (size_t)k * ldu;
    const bool keep = fabs(diag) >= fabs(sub);  // no row exchange
    const double piv = keep ? (fabs(diag) < tiny ? copysign(tiny, diag) : diag) : sub;
    const double rp = rcp_f64(piv);
    const double mlt = (keep ? sub : diag) * rp;
    const double p1 = keep ? sup : nd, p2 = keep ? 0.0 : ns, py = keep ? yk : yk1;
    const double o1 = keep ? nd : sup, o2 = keep ? ns : 0.0, oy = keep ? yk1 : yk;
    U0[o] = rp;
    U1[o] = p1;
    U2[o] = p2;
    z[k * ldz] = py;
    yk = fma(-mlt, py, oy);
    diag = fma(-mlt, p1, o1);
    sup = fma(-mlt, p2, o2);
  }
  const double rlast = 1.0 / (fabs(diag) < tiny ? copysign(tiny, diag) : diag);
  double x1 = yk * rlast, x2 = 0.0, xmax = fabs(x1);
  z[(n - 1) * ldz] = x1;
  // back substitution in blocks of kPF rows: the U factors of the next block are loaded while
  // this block is solved (the loads come from L2; one row ahead left each row waiting on one)
  constexpr int kPF = 8;
  double c0[kPF], c1[kPF], c2[kPF];
#pragma unroll
  for (int t = 0; t < kPF; ++t) {
    const int kk = n - 2 - t;
    const size_t o = (size_t)(kk >= 0 ? kk : 0) * ldu;
    c0[t] = U0[o];
    c1[t] = U1[o];
    c2[t] = U2[o];
  }
  for (int k0 = n - 2; k0 >= 0; k0 -= kPF) {
    double n0[kPF], n1[kPF], n2[kPF];
#pragma unroll
    for (int t = 0; t < kPF; ++t) {
      const int kk = k0 - kPF - t;
      const size_t o = (size_t)(kk >= 0 ? kk : 0) * ldu;
      n0[t] = U0[o];
      n1[t] = U1[o];
      n2[t] = U2[o];
    }
#pragma unroll
    for (int t = 0; t < kPF; ++t) {
      const int k = k0 - t;
      if (k >= 0) {
        const double x = (z[k * ldz] - c1[t] * x1 - c2[t] * x2) * c0[t];
        z[k * ldz] = x;
        xmax = fmax(xmax, fabs(x));
        x2 = x1;
        x1 = x;
      }
    }
#pragma unroll
    for (int t = 0; t < kPF; ++t) {
      c0[t] = n0[t];
      c1[t] = n1[t];
      c2[t] = n2[t];
    }
  }
  const double sc = xmax > 0.0 ? 1.0 / xmax : 1.0;
  double nrm = 0.0;
  for (int k = 0; k < n; ++k) {
    const double v = z[k * ldz] * sc;
    z[k * ldz] = v;
    nrm = fma(v, v, nrm);
  }
  return nrm > 0.0 ? 1.0 / sqrt(nrm) : 0.0;
}

// ---- the thread grid of the Householder phase.  The lanes of a wave form 4 rows x 16 columns:
// column tc = lane bits 5 4 1 0, row rl = lane bits 3 2; thread row tr = 4 wave + rl.
// Sum over the 16 columns of a thread row: the two high bits by permlane swaps, the two low ones by
// quad permutations (VALU only).  Every lane of the row ends with the same bits.
__device__ inline double cols16_sum(double v) {
  v = swap32_sum(v);
  v = swap16_sum(v);
  v += dpp_f64<0xB1>(v);
  v += dpp_f64<0x4E>(v);
  return v;
}
// lanes 0-31: the sum over bit 5 of a; lanes 32-63: of b
__device__ inline double fold32(double a, double b) {
  const unsigned long long x = (unsigned long long)__double_as_longlong(a);
  const unsigned long long y = (unsigned long long)__double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  return __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0])) +
         __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
}
// lanes with bit 4 clear: the sum over bit 4 of a; set: of b
__device__ inline double fold16(double a, double b) {
  const unsigned long long x = (unsigned long long)__double_as_longlong(a);
  const unsigned long long y = (unsigned long long)__double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  return __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0])) +
         __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
}

// Workgroup barrier for LDS alone: the reflector stores to the workspace stay in flight (a full
// barrier waits for each of them).  One wave needs none: its LDS accesses execute in order.
template <int NW>
__device__ inline void lds_barrier() {
  if constexpr (NW == 1)
    asm volatile("" ::: "memory");
  else
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

struct TriState {
  double* xb;   // reflector column, S rows (LDS)
  double* pb;   // p = tau A u, S rows (LDS)
  double2* de;  // diagonal in .x
  double* e;
  double* tau;
  double* HH;  // reflectors, row i - off, column c - off
  int off, nmax, tr, tc, lane, wave;
};

// Householder steps whose first live row j lies in row slot A0 (so that slots below A0, rows and
// columns alike, are finished: their work is left out at compile time), then those of A0 + 1.
//
// Step j eliminates column j - 1.  x = A[j:, j-1] is in LDS (zero below row j).  With
// beta = -sign(x_j) |x| and u = x - beta e_j: H = I - tau u u^T, tau = 1 / (|x|^2 + |x_j| |x|),
// p = tau A u, w = p - (tau / 2)(p.u) u, A -= u w^T + w u^T.  The vectors need no scaling pass, and
// A u = A x - beta A[:, j] starts before beta is known.  Two barriers per step: x, then p.  Every
// wave holds all columns of x and p, so |x|^2 and p.u are summed in each wave without LDS.
// What bounds it: instruction issue and the latency of this chain, not arithmetic (a wave's
// vector instruction takes 4 cycles whatever it does), hence the few instructions per step:
// row sums folded two values at a time by permlane swaps, no range tests (the block sits at the
// high end of the grid, rows and columns below `off` are zero), column j updated first.  One block of
// 182 orbitals: 630 -> 235 us; of 92 (4 waves) 210 -> 71; of 14 (one wave) 34 -> 8.
template <int NW, int RR, int RC, int A0>
__device__ __forceinline__ void tri_steps(double (&A)[RR][RC], int& j, const TriState& t) {
  constexpr int GR = 4 * NW, S = GR * RR;
  constexpr int B0 = A0 * GR / 16, B1 = ((A0 + 1) * GR - 1) / 16;  // column slots that may hold j
  constexpr int R = RR - A0, C = RC - B0;
  constexpr int R1 = (R + 1) / 2, R2 = (R1 + 1) / 2;  // row sums left after each fold
  const int last = min((A0 + 1) * GR - 1, S - 2);
  const int b5 = t.lane >> 5, b4 = (t.lane >> 4) & 1, quad = t.lane & 3;
  // quad lane q writes folded value q: row slot of that value in this lane
  const int i1 = min(2 * min(quad, R2 - 1) + b4, R1 - 1);
  const int prow = (A0 + min(2 * i1 + b5, R - 1)) * GR + t.tr;
  const double* xcol = t.xb + t.tc + 16 * B0;
  const double* xrow = t.xb + t.tr + GR * A0;
  const double* pcol = t.pb + t.tc + 16 * B0;
  const double* prw = t.pb + t.tr + GR * A0;
  for (; j <= last; ++j) {
    lds_barrier<NW>();
    double uc[C], ur[R];
#pragma unroll
    for (int b = 0; b < C; ++b) uc[b] = xcol[16 * b];
#pragma unroll
    for (int a = 0; a < R; ++a) ur[a] = xrow[GR * a];
    const double alpha = t.xb[j];
    double s[R];
#pragma unroll
    for (int a = 0; a < R; ++a) s[a] = 0.0;
#pragma unroll
    for (int b = 0; b < C; ++b)
#pragma unroll
      for (int a = 0; a < R; ++a) s[a] = fma(A[A0 + a][B0 + b], uc[b], s[a]);
    double q0 = 0.0, q1 = 0.0;
#pragma unroll
    for (int b = 0; b < C; ++b) {
      if (b & 1)
        q1 = fma(uc[b], uc[b], q1);
      else
        q0 = fma(uc[b], uc[b], q0);
    }
    const double x2 = cols16_sum(q0 + q1);
    double tau = 0.0, beta = alpha;
    if (!(x2 <= 1.0e-280)) {  // |x| below 1e-140 counts as zero; a NaN goes on
      double r = __builtin_amdgcn_rsq(x2);
      r = fma(0.5 * r, fma(-x2 * r, r, 1.0), r);
      r = fma(0.5 * r, fma(-x2 * r, r, 1.0), r);
      double nx = x2 * r;
      nx = fma(0.5 * r, fma(-nx, nx, x2), nx);
      beta = -copysign(nx, alpha);
      tau = rcp_f64(fma(fabs(alpha), nx, x2));
    }
    // x -> u, and the sums' share of it
    const double pt = t.tc == (j & 15) ? -beta : 0.0;
    const int bn = j >> 4;
#pragma unroll
    for (int b = B0; b <= B1; ++b)
      if (b == bn) {  // uniform
#pragma unroll
        for (int a = 0; a < R; ++a) s[a] = fma(A[A0 + a][b], pt, s[a]);
        uc[b - B0] += pt;
      }
    ur[0] += t.tr + GR * A0 == j ? -beta : 0.0;
    // row sums: fold over column bit 5, then 4, then sum over the quad
    double f[R1], g[R2];
#pragma unroll
    for (int i = 0; i < R1; ++i) f[i] = fold32(s[2 * i], s[min(2 * i + 1, R - 1)]);
#pragma unroll
    for (int i = 0; i < R2; ++i) {
      g[i] = fold16(f[2 * i], f[min(2 * i + 1, R1 - 1)]);
      g[i] += dpp_f64<0xB1>(g[i]);
      g[i] += dpp_f64<0x4E>(g[i]);
    }
    double pval = g[0];
#pragma unroll
    for (int i = 1; i < R2; ++i) pval = quad == i ? g[i] : pval;
    if (quad < R2) t.pb[prow] = prow >= j ? tau * pval : 0.0;
    if (t.wave == j % NW && (t.lane & 12) == 0) {  // one wave stores u
      double* h = t.HH + (size_t)(j - 1 - t.off) * t.nmax - t.off + t.tc + 16 * B0;
#pragma unroll
      for (int b = 0; b < C; ++b)
        if (b > B1 - B0 || t.tc + 16 * (B0 + b) >= j) h[16 * b] = uc[b];
      if (t.lane == 0) {
        t.e[j - 1 - t.off] = beta;
        t.tau[j - 1 - t.off] = tau;
      }
    }
    lds_barrier<NW>();
    double wc[C], wr[R];
#pragma unroll
    for (int b = 0; b < C; ++b) wc[b] = pcol[16 * b];
#pragma unroll
    for (int a = 0; a < R; ++a) wr[a] = prw[GR * a];
    q0 = q1 = 0.0;
#pragma unroll
    for (int b = 0; b < C; ++b) {
      if (b & 1)
        q1 = fma(uc[b], wc[b], q1);
      else
        q0 = fma(uc[b], wc[b], q0);
    }
    const double K = -0.5 * tau * cols16_sum(q0 + q1);
#pragma unroll
    for (int a = 0; a < R; ++a) wr[a] = fma(K, ur[a], wr[a]);
#pragma unroll
    for (int b = 0; b < C; ++b) {
      const double wb = fma(K, uc[b], wc[b]);
#pragma unroll
      for (int a = 0; a < R; ++a) A[A0 + a][B0 + b] = fma(-ur[a], wb, fma(-wr[a], uc[b], A[A0 + a][B0 + b]));
      if (b <= B1 - B0 && B0 + b == bn && t.tc == (j & 15)) {  // column j: the next x, and d_j
#pragma unroll
        for (int a = 0; a < R; ++a) {
          const double val = A[A0 + a][B0 + b];
          if (a == 0) {
            const int r = t.tr + GR * A0;
            t.xb[r] = r > j ? val : 0.0;
            if (r == j) t.de[j - t.off].x = val;
          } else {
            t.xb[t.tr + GR * (A0 + a)] = val;
          }
        }
      }
    }
  }
  if constexpr (A0 + 1 < RR) tri_steps<NW, RR, RC, A0 + 1>(A, j, t);
}

// Householder tridiagonalisation of the n x n block Fm, held in registers at the high end of the
// S x S grid: thread (tr, tc) holds A[tr + GR a][tc + 16 b], a < RR, b < RC, row r of the grid being
// row r - off of the block.
template <int NW, int RR, int RC>
__device__ __forceinline__ void tridiagonalise(const double* __restrict__ Fm, int n, const TriState& t) {
  constexpr int GR = 4 * NW, S = GR * RR, NT = 64 * NW;
  static_assert(16 * RC == S, "square register grid");
  double A[RR][RC];
#pragma unroll
  for (int a = 0; a < RR; ++a)
#pragma unroll
    for (int b = 0; b < RC; ++b) {
      const int r = t.tr + GR * a - t.off, c = t.tc + 16 * b - t.off;
      A[a][b] = (r >= 0 && c >= 0) ? Fm[(size_t)r * n + c] : 0.0;
    }
  // reflector i is zero at the columns <= i of its panel
  for (int k = threadIdx.x; k < n * 16; k += NT) {
    const int i = k / 16 + t.off, c = (i & ~15) + (k & 15);
    if (c <= i && c >= t.off) t.HH[(size_t)(i - t.off) * t.nmax + c - t.off] = 0.0;
  }
#pragma unroll
  for (int b = 0; b < RC; ++b)
    if (b == t.off / 16 && t.tc == (t.off & 15)) {
#pragma unroll
      for (int a = 0; a < RR; ++a) {
        const int r = t.tr + GR * a;
        t.xb[r] = r > t.off ? A[a][b] : 0.0;
        if (r == t.off) t.de[0].x = A[a][b];
      }
    }
  int j = t.off + 1;
  tri_steps<NW, RR, RC, 0>(A, j, t);
  lds_barrier<NW>();
  if (n >= 2 && t.tr == GR - 1 && t.tc == 15) {
    t.e[n - 2] = t.xb[S - 1];
    t.de[n - 1].x = A[RR - 1][RC - 1];
  }
  __syncthreads();
}

// T of the block reflector H_16q ... H_16q+15 = I - V T V^T (V's columns the reflectors u of panel
// q), T = (diag(1/tau) + strict upper triangle of V^T V)^-1, by back substitution: lane c of the
// wave computes column c.  Written row-major to Tq.  Reflectors outside off .. S - 3 have tau = 0.
template <int S>
__device__ void panel_t(const double* __restrict__ HH, const double* tau, int nmax, int n, int q, double* Tq) {
  const int off = S - n, lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
  const int refl = min(max(16 * q + m - off, 0), n - 3);
  const double* v = HH + (size_t)refl * nmax;
  doublex4 G = {0.0, 0.0, 0.0, 0.0};
  for (int r = 16 * q; r < S; r += 16) {
    double a[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int c = r + 4 * s + g - off;
      a[s] = c >= 0 ? v[c] : 0.0;
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) G = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], a[s], G, 0, 0, 0);
  }
  // G[r][c] sits in register r / 4 of lane 16 (r % 4) + c
  const int im = 16 * q + m - off;
  const double tm = (im >= 0 && im <= n - 3) ? tau[im] : 0.0;
  double T[16];
#pragma unroll
  for (int i = 15; i >= 0; --i) {
    double acc = 0.0;
#pragma unroll
    for (int k = i + 1; k < 16; ++k) {
      const long long w = __double_as_longlong(G[i >> 2]);
      const int src = 16 * (i & 3) + k;
      const unsigned lo = __builtin_amdgcn_readlane((int)w, src), hi = __builtin_amdgcn_readlane((int)(w >> 32), src);
      acc = fma(__longlong_as_double(((long long)hi << 32) | lo), T[k], acc);
    }
    const long long w = __double_as_longlong(tm);
    const unsigned lo = __builtin_amdgcn_readlane((int)w, i), hi = __builtin_amdgcn_readlane((int)(w >> 32), i);
    const double ti = __longlong_as_double(((long long)hi << 32) | lo);
    T[i] = m == i ? ti : (m > i ? -ti * acc : 0.0);
  }
  if (g == 0) {
#pragma unroll
    for (int i = 0; i < 16; ++i) Tq[16 * i + m] = T[i];
  }
}

// Panels q, q - 1, ..., 0 of the back-transformation on one wave's 16 columns of Z: C -= V T V^T C.
// Cr[t] holds rows 16 t + 4 s + lane / 16 (element s), column lane % 16: the MFMA result layout,
// which is also the layout of its right operand, so C needs no move between the three products.
// V and T come from the workspace (the waves read the same panel: L1 / L2).  One reflector at a
// time on vector instructions took 201 us for 91 vectors of 182 orbitals (each step waited for its
// reflector); blocks of 16 take 71 us, bounded by those reads and the chain of products.
template <int S, int Q>
__device__ __forceinline__ void back_panels(doublex4 (&Cr)[S / 16], const double* __restrict__ HH,
                                            const double* __restrict__ T, int nmax, int n) {
  constexpr int NTL = S / 16;
  const int off = S - n;
  if (16 * Q + 15 >= off) {  // uniform
    int m = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    asm volatile("" : "+v"(m), "+v"(g));  // keeps every panel's addresses from being held at once (they spill)
    // V's operands are read one tile ahead of their products; the scheduler, left alone, reads whole
    // panels ahead and spills
    const int o1 = min(max(16 * Q + m - off, 0), n - 3) * nmax - off + g;
    int o2[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) o2[s] = min(max(16 * Q + 4 * s + g - off, 0), n - 3) * nmax - off + m;
    const double* tq = T + kTPanel * Q + 16 * m + g;
    doublex4 y0 = {0.0, 0.0, 0.0, 0.0}, y1 = {0.0, 0.0, 0.0, 0.0};
    double a[2][4], tv[4];
    // rows below off (first tile only) are zero in C; their V is read at the block's first row
#pragma unroll
    for (int s = 0; s < 4; ++s) a[0][s] = HH[o1 + max(16 * Q + 4 * s, off - g)];
#pragma unroll
    for (int t = Q; t < NTL; ++t) {
      const int k = (t - Q) & 1;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (t + 1 < NTL)
          a[k ^ 1][s] = HH[o1 + 16 * t + 16 + 4 * s];
        else
          tv[s] = tq[4 * s];
      }
      y0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[k][0], Cr[t][0], y0, 0, 0, 0);
      y1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[k][1], Cr[t][1], y1, 0, 0, 0);
      y0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[k][2], Cr[t][2], y0, 0, 0, 0);
      y1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[k][3], Cr[t][3], y1, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) a[0][s] = HH[o2[s] + max(16 * Q, off - m)];
    y0 += y1;
    doublex4 y = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < 4; ++s) y = __builtin_amdgcn_mfma_f64_16x16x4f64(-tv[s], y0[s], y, 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = Q; t < NTL; ++t) {
      const int k = (t - Q) & 1;
      if (t + 1 < NTL) {
#pragma unroll
        for (int s = 0; s < 4; ++s) a[k ^ 1][s] = HH[o2[s] + 16 * t + 16];
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) Cr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[k][s], y[s], Cr[t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if constexpr (Q > 0) back_panels<S, Q - 1>(Cr, HH, T, nmax, n);
}

// EVEC = false: the density P = 2 C_occ C_occ^T of the nocc lowest vectors.  EVEC = true: every
// eigenpair (nv = n vectors), written as Qout (packed layout, column j = eigenvector j) and evals
// (orb_off[m] + j, the Rayleigh quotients of the final vectors: exact to rounding whatever the
// multisection bracket width).  GZ: the vectors stand in memory instead of LDS, for blocks whose vectors
// do not fit (all of 140 to 192 orbitals, or the occupied ones of clusters where they are most of the
// basis): with EVEC in Qout itself, else in zbuf (nmax^2 doubles per slot).  Rows are read ahead of their
// use in every sweep, and lanes run along a row, so the L2 serves them.
// Errors of all eigenpairs, 14 to 192 orbitals, against extended precision (the library's batched solver on the
// same blocks in brackets): energies 4.5e-16 of the largest [5.7e-16], squared vector elements of random
// spectra 2.5e-14 to 5.7e-13 [1.1e-13 to 1.0e-12], of alkane Fock matrices 0.8e-14 to 1.4e-13 [1.2e-14
// to 1.3e-13]; vectors orthogonal to 1e-14 to 6e-14 [2e-15 to 3e-15], residuals 4e-16 to 7e-16 |F|.
// All pairs of 128 alkanes of 2-30 carbons: 0.72 ms for the blocks above 139 orbitals, 0.44 for the rest
// (6.5 ms by the library's batched solver on padded stacks).
// WPS: waves per SIMD the registers are held to (launch_eigh).
template <int NW, int RR, int RC, bool EVEC, bool GZ, int WPS>
__global__ __launch_bounds__(64 * NW, WPS) void k_eigh_density(pyseqm_layout_t L, const int* __restrict__ idx,
                                                       const double* __restrict__ F, double* __restrict__ P,
                                                       double* __restrict__ ws, int nmax,
                                                       int* __restrict__ fail, const long long* __restrict__ orb_off,
                                                       double* __restrict__ evals, double* __restrict__ zbuf) {
  constexpr int NT = 64 * NW, S = 16 * RC;
  extern __shared__ __align__(16) double lds[];
  const int slot = blockIdx.x;
  const int m = idx[slot];
  const int n = L.mol_norb[m];
  const int nv = EVEC ? n : L.mol_nocc[m];  // vectors computed
  const size_t mo = L.mol_mat_off[m];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const size_t nm2 = (size_t)nmax * nmax;
  double* HH = ws + (size_t)slot * 4 * nm2;
  double* U0 = HH + nm2;
  double* U1 = HH + 2 * nm2;
  double* U2 = HH + 3 * nm2;
  const int ldz = GZ ? nv : zstride(n, nv);
  double* Z = GZ ? (EVEC ? P + mo : zbuf + (size_t)slot * nm2) : lds;  // eigenvectors: Z[k * ldz + j]
  double2* de = reinterpret_cast<double2*>(lds + ((zregion(GZ ? 0 : n, nv, S) + 1) & ~1));  // (d, e^2)
  double* e = reinterpret_cast<double*>(de + n);
  double* lam = e + n;
  double* tau = lam + n;
  double* aux = tau + n;  // block reductions' scratch; the vectors' scales
  double* red = aux;
  unsigned char* twist = reinterpret_cast<unsigned char*>(aux + n);
  double* T = S == 48 ? aux + n + 24 : U0;  // the panels' T factors (and the lower multipliers after them)

  // ---- 1. tridiagonal form
  {
    TriState t;
    t.xb = lds;
    t.pb = lds + S;
    t.de = de;
    t.e = e;
    t.tau = tau;
    t.HH = HH;
    t.off = S - n;
    t.nmax = nmax;
    t.tc = (lane & 3) | ((lane >> 4) << 2);
    t.tr = 4 * wave + ((lane >> 2) & 3);
    t.lane = lane;
    t.wave = wave;
    tridiagonalise<NW, RR, RC>(F + mo, n, t);
  }
  // ---- 2. the nv lowest eigenvalues, and the next one above (its distance says how sharp the
  //         highest of them has to be).  What bounds it: instruction issue, some 7 per row and
  //         point, so the rounds after the grid run one wave per SIMD.  91 of 182: 144 -> 73 us
  const int nvx = EVEC ? n : min(nv + 1, n);
  double lo_p = 1.0e300, hi_p = -1.0e300;
  for (int k = tid; k < n; k += NT) {
    const double el = k > 0 ? fabs(e[k - 1]) : 0.0, er = k + 1 < n ? fabs(e[k]) : 0.0;
    lo_p = fmin(lo_p, de[k].x - el - er);
    hi_p = fmax(hi_p, de[k].x + el + er);
  }
  double glo = eig_block_min<NT>(lo_p, red);
  double ghi = eig_block_max<NT>(hi_p, red);
  const double tnorm = fmax(fabs(glo), fabs(ghi));
  const double slack = 2.2e-16 * tnorm * 4.0 + 2.0e-300 * fmax(1.0, tnorm);
  glo -= slack;
  ghi += slack;
  for (int k = tid; k + 1 < n; k += NT) de[k].y = fmax(e[k] * e[k], fmax(1.0e-60 * tnorm * tnorm, 1.0e-300));
  __syncthreads();
  const double btol = 1.0e-11 * tnorm, ctol = 1.0e-6 * tnorm, dtol = 1.0e-10 * tnorm, gtol = 1.0e-3 * tnorm;
  {
    constexpr int M = 2 * NT;  // grid points
    int* counts = reinterpret_cast<int*>(lds);
    const double step = (ghi - glo) / (double)(M + 1);
    {
      const double x[2] = {fma((double)(tid + 1), step, glo), fma((double)(tid + NT + 1), step, glo)};
      int c[2];
      sturm_counts<2>(de, n, x, c);
      counts[tid] = c[0];
      counts[tid + NT] = c[1];
    }
    __syncthreads();
    constexpr int kLanes = NT > 256 ? 256 : NT;  // one wave per SIMD
    int tb = 64;
    while (tb > 1 && nvx * tb > kLanes) tb >>= 1;  // nvx <= NT in every variant
    const int j = tid / tb, gl = tid % tb;
    double lo = glo, hi = ghi;
    auto narrow = [&](double tol) {  // uniform over the lane group
      for (int round = 0; round < 64; ++round) {
        if (!(hi - lo > fmax(4.4e-16 * fmax(fabs(lo), fabs(hi)), tol) + 2.0e-300)) break;
        const double x[1] = {lo + (hi - lo) * (double)(gl + 1) / (double)(tb + 1)};
        int c[1];
        sturm_counts<1>(de, n, x, c);
        const bool in = x[0] > lo && x[0] < hi;
        const double nlo = group_max_t(in && c[0] <= j ? x[0] : lo, tb);
        const double nhi = group_min_t(in && c[0] > j ? x[0] : hi, tb);
        if (nlo == lo && nhi == hi) break;  // no representable interior point left
        lo = nlo;
        hi = nhi;
      }
    };
    if (j < nvx) {
      int a = -1, b = M;  // counts[a] <= j < counts[b]
      while (b - a > 1) {
        const int c = (a + b) >> 1;
        if (counts[c] > j)
          b = c;
        else
          a = c;
      }
      if (a >= 0) lo = fma((double)(a + 1), step, glo);
      if (b < M) hi = fma((double)(b + 1), step, glo);
      narrow(btol);
      if (gl == 0) lam[j] = 0.5 * (lo + hi);
    }
    __syncthreads();
    // A bracket b leaves the Rayleigh correction b^2 / gap off, and the vector that over the other gaps: where a
    // neighbour is closer than ctol the bracket shrinks until that is below 1e-16 |T|.
    double gap = 2.0 * ctol;
    if (j < nvx && j > 0) gap = fmin(gap, lam[j] - lam[j - 1]);
    if (j + 1 < nvx) gap = fmin(gap, lam[j + 1] - lam[j]);
    __syncthreads();
    if (gap <= ctol) {
      narrow(gap <= 1.0e-9 * tnorm ? 0.0 : 1.0e-8 * sqrt(gap * tnorm));
      if (gl == 0) lam[j] = 0.5 * (lo + hi);
    }
    __syncthreads();
  }
  // e^2 is done with: .y carries the part of each eigenvalue below lam's rounding
  for (int k = tid; k < n; k += NT) de[k].y = 0.0;
  auto degenerate = [&](int j) {
    return (j > 0 && lam[j] - lam[j - 1] <= dtol) || (j + 1 < nvx && lam[j + 1] - lam[j] <= dtol);
  };
  const bool mine = tid < nv && degenerate(tid);  // nv <= NT in every variant
  const bool any_degenerate = __syncthreads_or(mine);

  // ---- 3. eigenvectors: NT / 2 vectors at a time, lane `side` 0 from the top, 1 from the bottom.
  // L and U: the two ends' multipliers (twisted_sweep).  The twist row r has the least |gamma_k|, gamma_k =
  // d_k - lambda - e_{k-1} L_{k-1} - e_k U_k.  z_r = 1, outwards z = -L z (products only), and gamma_r / |z|^2
  // corrects lambda.  Kept unrounded as lam + .y: rounded, it would tilt the vectors of neighbours at a
  // gap by eps |T| / gap.
  constexpr int kHalf = NT / 2;
  {
    // waves 0 1 and 2 3 (a SIMD each), then 4 5 and 6 7; the halves of a lone wave
    const int side = NW == 1 ? lane >> 5 : (wave >> 1) & 1;
    const int vec = NW == 1 ? lane & 31 : lane + 64 * ((wave & 1) + 2 * (wave >> 2));
    double* U = S == 48 ? T + 3 * kTPanel : U0;
    const int ldu = S == 48 ? ldz : nmax;
    const double tiny = 1.0e-40 * fmax(tnorm, 1.0e-200);
    // levels degenerate to rounding keep their bisected eigenvalue: a twisted vector of theirs may be poor
    static_assert(2 * kHalf >= S, "a thread has at most two vectors");
    const bool keep[2] = {vec < nv && degenerate(vec), kHalf + vec < nv && degenerate(kHalf + vec)};
    for (int c0 = 0; c0 < nv; c0 += kHalf) {
      const int j = c0 + vec;
      const int nc = min(kHalf, nv - c0);
      const bool live = j < nv;
      int r = 0;  // the twist row, of the first factorisation for both
      for (int pass = 0; pass < 2; ++pass) {
        if (live) {
          const double hi = lam[j], lo = de[j].y;
          if (side == 0)
            twisted_sweep<1>(de, e, n, hi, lo, tiny, Z + j, ldz);
          else
            twisted_sweep<-1>(de + n - 1, e + n - 2, n, hi, lo, tiny, U + (n - 2) * ldu + j, -ldu);
        }
        __syncthreads();
        double gam = 0.0;
        if (pass == 0) {  // twist rows: tg lanes per vector, rows part, part + tg, ...
          int tg = 64;
          while (nc * tg > NT) tg >>= 1;
          const int v = tid / tg, part = tid % tg, jv = c0 + v;
          if (v < nc) {
            const double hi = lam[jv], lo = de[jv].y;
            double best = 0.0;
            int rb = -1;
            auto take = [&](double g, int k) {
              if (rb < 0 || fabs(g) < fabs(best)) {
                best = g;
                rb = k;
              }
            };
            const double* zl = Z + jv - ldz;
            const double* ul = U + jv;
            int k = part;
            if (k == 0) {
              take(n > 1 ? fma(-e[0], ul[0], (de[0].x - hi) - lo) : (de[0].x - hi) - lo, 0);
              k += tg;
            }
#pragma unroll 4
            for (; k + 1 < n; k += tg)
              take(fma(-e[k], ul[k * ldu], fma(-e[k - 1], zl[k * ldz], (de[k].x - hi) - lo)), k);
            if (k + 1 == n) take(fma(-e[k - 1], zl[k * ldz], (de[k].x - hi) - lo), k);
            for (int o = 1; o < tg; o <<= 1) {
              const double og = __shfl_xor(best, o);
              const int orow = __shfl_xor(rb, o);
              if (orow >= 0 && (rb < 0 || fabs(og) < fabs(best) || (fabs(og) == fabs(best) && orow < rb))) {
                best = og;
                rb = orow;
              }
            }
            if (part == 0) {
              aux[jv] = best;
              twist[jv] = (unsigned char)max(rb, 0);
            }
          }
          __syncthreads();
          if (live) {
            gam = aux[j];
            r = twist[j];
          }
          __syncthreads();  // every lane has its gamma: aux takes the norms
        }
        double nrm = 0.0;
        if (live) {
          double z = 0.0;
          if (side == 0) {
            // rows up to the twist row only, read and written: the other wave writes those beyond it meanwhile
            const int zr = r * ldz + j;
            auto row = [&](double* zk, double l, int k) {
              z = k == r ? 1.0 : -l * z;  // zero above the twist row, until it
              if (k <= r) {
                *zk = z;
                nrm = fma(z, z, nrm);
              }
            };
            const int n8 = n & ~7;
            if (n > n8) row(Z + (n - 1) * ldz + j, 0.0, n - 1);
            for (int k = n - 2; k >= n8; --k) row(Z + k * ldz + j, Z[min(k * ldz + j, zr)], k);
            if (n8) {
              int zk = (n8 - 8) * ldz + j;
              double l[8];
#pragma unroll
              for (int t = 0; t < 8; ++t) l[t] = Z[min(zk + t * ldz, zr)];
              if (n8 == n) l[7] = 0.0;  // row n - 1 has no multiplier
#pragma unroll 2
              for (int k0 = n8 - 8; k0 >= 0; k0 -= 8) {
                double ln[8];
                if (k0 >= 8) {
#pragma unroll
                  for (int t = 0; t < 8; ++t) ln[t] = Z[min(zk + (t - 8) * ldz, zr)];
                }
#pragma unroll
                for (int t = 7; t >= 0; --t) row(Z + zk + t * ldz, l[t], k0 + t);
#pragma unroll
                for (int t = 0; t < 8; ++t) l[t] = ln[t];
                zk -= 8 * ldz;
              }
            }
            aux[j] = nrm;
          } else {
            auto row = [&](double* zk, double u, int k) {
              z = k == r ? 1.0 : -u * z;
              if (k > r) {
                *zk = z;
                nrm = fma(z, z, nrm);
              }
            };
            if (r == 0) z = 1.0;
            constexpr int kB = 16;  // the multipliers come from the workspace (L2): rows read ahead
            double* zk = Z + ldz + j;
            const double* uk = U + j;
            int k0 = 1;
            if (n > kB) {
              double u[kB];
#pragma unroll
              for (int t = 0; t < kB; ++t) u[t] = uk[t * ldu];
#pragma unroll 2
              for (; k0 + kB <= n; k0 += kB) {
                double un[kB];
                if (k0 + 2 * kB <= n) {
#pragma unroll
                  for (int t = 0; t < kB; ++t) un[t] = uk[(kB + t) * ldu];
                }
#pragma unroll
                for (int t = 0; t < kB; ++t) row(zk + t * ldz, u[t], k0 + t);
#pragma unroll
                for (int t = 0; t < kB; ++t) u[t] = un[t];
                zk += kB * ldz;
                uk += kB * ldu;
              }
            }
#pragma unroll 4
            for (; k0 < n; ++k0) {
              row(zk, *uk, k0);
              zk += ldz;
              uk += ldu;
            }
          }
        }
        __syncthreads();
        if (live && side == 1) {
          nrm += aux[j];
          aux[j] = 1.0 / sqrt(nrm);  // the vector's scale
          if (pass == 0 && !keep[c0 > 0]) {
            const double corr = fmin(fmax(gam / nrm, -btol), btol);
            const double s = lam[j] + corr;
            de[j].y = corr - (s - lam[j]);
            lam[j] = s;
          }
        }
        __syncthreads();
      }
    }
  }
  // Vectors of degenerate levels (pass 0 and 1): two solves from different starts, orthogonalised within
  // the level, one more solve, orthogonalised again.  At shifts equal to rounding a solve may favour one
  // vector of the level a hundredfold, so that two starts come out nearly parallel; what the first
  // orthogonalisation leaves of the second is small and carries the error of the rest of the spectrum
  // magnified, which the third solve takes out again.  Density errors at such levels (8 to 192
  // orbitals): 1e-14 to 1e-12; with three solves and one orthogonalisation after them up to 1e-10.
  // ---- 4. clusters (runs of eigenvalues closer than gtol; pass 2): chain after chain per wave, each vector
  //         against those before it within gtol, four at a time (their products are small, so that is
  //         the same to rounding as one by one); a second time where it lost half of its length.
  //         182 orbitals: 15-61 us by one thread per cluster at 1e-5 |T|, 13-26 here at 1e-3
  for (int pass = any_degenerate ? 0 : 2; pass < 3; ++pass) {
    const double tol = pass < 2 ? dtol : gtol;
    if (pass < 2) {
      const double tiny = 2.2e-16 * fmax(tnorm, 1.0e-300);
      for (int solve = pass; mine && solve < 2; ++solve)
        aux[tid] = inverse_iteration(de, e, Z + tid, ldz, U0 + tid, U1 + tid, U2 + tid, nmax, n, tid, lam[tid], tiny,
                                     pass + solve == 0);
      __syncthreads();
    }
    constexpr int E = (S + 63) / 64;
    int chain = 0;
    for (int base = 0; base < nv; base += 64) {
      const int jl = base + lane;
      const bool starts = jl + 1 < nv && (jl == 0 || lam[jl] - lam[jl - 1] > tol) && lam[jl + 1] - lam[jl] <= tol;
      unsigned long long todo = __ballot(starts);
      for (; todo; todo &= todo - 1, ++chain) {
        if (chain % NW != wave) continue;
        const int first = base + __ffsll(todo) - 1;
        int p0 = first;
        for (int q = first; q < nv && (q == first || lam[q] - lam[q - 1] <= tol); ++q) {
          double zq[E];
          const double sc = aux[q];
#pragma unroll
          for (int i = 0; i < E; ++i) {
            const int k = lane + 64 * i;
            zq[i] = k < n ? sc * Z[k * ldz + q] : 0.0;
          }
          while (lam[q] - lam[p0] > tol) ++p0;
          for (int rep = 0; rep < 2; ++rep) {
            for (int p = p0; p < q; p += 4) {
              double zp[4][E], dot[4];
#pragma unroll
              for (int c = 0; c < 4; ++c) {
                dot[c] = 0.0;
#pragma unroll
                for (int i = 0; i < E; ++i) {
                  const int k = lane + 64 * i;
                  zp[c][i] = k < n && p + c < q ? Z[min(k, n - 1) * ldz + min(p + c, q)] : 0.0;
                  dot[c] = fma(zp[c][i], zq[i], dot[c]);
                }
              }
#pragma unroll
              for (int c = 0; c < 4; ++c) dot[c] = wave64(dot[c]);
#pragma unroll
              for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int i = 0; i < E; ++i) zq[i] = fma(-dot[c], zp[c][i], zq[i]);
            }
            double nr = 0.0;
#pragma unroll
            for (int i = 0; i < E; ++i) nr = fma(zq[i], zq[i], nr);
            nr = wave64(nr);
            if (!(nr > 1.0e-200)) {  // lost to its cluster's span: flagged, left unscaled
              if (lane == 0 && pass == 2) atomicAdd(fail, 1);
              break;
            }
            const double s = 1.0 / sqrt(nr);
#pragma unroll
            for (int i = 0; i < E; ++i) zq[i] *= s;
            if (nr > 0.5) break;
          }
#pragma unroll
          for (int i = 0; i < E; ++i) {
            const int k = lane + 64 * i;
            if (k < n) Z[k * ldz + q] = zq[i];
          }
          if (lane == 0) aux[q] = 1.0;
        }
      }
    }
    __syncthreads();
  }

  if (EVEC) {
    // Rayleigh quotients of the vectors as lam + z^T (T - lam) z / z^T z, a group of
    // lanes per vector: the rows of (T - lam) z are residuals, so their sum rounds at the size of those and not of T
    int tg = 64;
    while (nv * tg > NT) tg >>= 1;
    const int j = tid / tg;
    const double s = lam[min(j, nv - 1)];
    double acc = 0.0;
    if (j < nv)
      for (int k = tid % tg; k < n; k += tg) {
        const double* z = Z + k * ldz + j;
        double row = (de[k].x - s) * z[0];
        if (k > 0) row = fma(e[k - 1], z[-ldz], row);
        if (k + 1 < n) row = fma(e[k], z[ldz], row);
        acc = fma(z[0], row, acc);
      }
    acc = group_sum_t(acc, tg);
    if (j < nv && tid % tg == 0) lam[j] = s + acc * aux[j] * aux[j];
    __syncthreads();
  }
  // ---- 5. C = Q Z: 16 columns per wave in registers, blocks of 16 reflectors last to first, each
  //         as C -= V (T (V^T C)) on FP64 MFMA; C goes back over Z
  if (n >= 3) {
    constexpr int NTL = S / 16;
    for (int q = wave + (S - n) / 16; q < NTL; q += NW) panel_t<S>(HH, tau, nmax, n, q, T + kTPanel * q);
    __syncthreads();
    const int off = S - n;
    for (int vt = wave; 16 * vt < nv; vt += NW) {
      const int col = 16 * vt + (lane & 15), g = lane >> 4;
      const double scale = aux[min(col, nv - 1)];
      doublex4 Cr[NTL];
#pragma unroll
      for (int t = 0; t < NTL; ++t)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int k = 16 * t + 4 * s + g - off;
          const double z = Z[max(k, 0) * ldz + min(col, nv - 1)];
          Cr[t][s] = (k >= 0 && col < nv) ? z * scale : 0.0;
        }
      const double* hh = HH;
      const double* tt = T;
      asm volatile("" : "+s"(hh));  // keep the panels' loads inside the loop (hoisted, they spill)
      if constexpr (S != 48) asm volatile("" : "+s"(tt));
      back_panels<S, NTL - 1>(Cr, hh, tt, nmax, n);
#pragma unroll
      for (int t = 0; t < NTL; ++t)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int k = 16 * t + 4 * s + g - off;
          if (k >= 0 && col < nv) Z[k * ldz + col] = Cr[t][s];
        }
    }
    __syncthreads();
  } else {  // no reflectors
    for (int t = tid; t < n * nv; t += NT) Z[(t / nv) * ldz + t % nv] *= aux[t % nv];
    __syncthreads();
  }
  if (EVEC) {
    if (!GZ) {
      double* Qm = P + mo;
      for (int t = tid; t < n * n; t += NT) Qm[t] = Z[(t / n) * ldz + t % n];  // row = orbital, column = vector
    }
    for (int j = tid; j < n; j += NT) {  // ascending: the quotients of a degenerate level may differ by rounding
      double v = lam[j];
      for (int k = j - 1; k >= 0 && !(lam[j] - lam[k] > dtol); --k)
        if (lam[k] > v) v = lam[k];
      evals[orb_off[m] + j] = v;
    }
    return;
  }
  // ---- P = 2 C C^T, a 16 x 16 tile of the upper triangle per wave at a time (two chains over the
  //      vectors, added); elements r <= c are written to both triangles: the two copies are the
  //      same bits.  91 vectors of 182 orbitals: 58 us as 4 x 4 blocks per thread, 21 us as MFMA tiles
  double* Pm = P + mo;
  const int nt = (n + 15) / 16, ntask = nt * (nt + 1) / 2;
  const int mr = lane & 15, g = lane >> 4, nfull = nv / 4;
  for (int task = wave; task < ntask; task += NW) {
    int bi = 0, rem = task;
    while (rem >= nt - bi) {
      rem -= nt - bi;
      ++bi;
    }
    const int bj = bi + rem;
    const double* ca = Z + min(16 * bi + mr, n - 1) * ldz + g;
    const double* cb = Z + min(16 * bj + mr, n - 1) * ldz + g;
    doublex4 a0 = {0.0, 0.0, 0.0, 0.0}, a1 = {0.0, 0.0, 0.0, 0.0};
    int k = 0;
    for (; k + 1 < nfull; k += 2) {
      a0 = __builtin_amdgcn_mfma_f64_16x16x4f64(ca[4 * k], cb[4 * k], a0, 0, 0, 0);
      a1 = __builtin_amdgcn_mfma_f64_16x16x4f64(ca[4 * k + 4], cb[4 * k + 4], a1, 0, 0, 0);
    }
    if (k < nfull) a0 = __builtin_amdgcn_mfma_f64_16x16x4f64(ca[4 * k], cb[4 * k], a0, 0, 0, 0);
    if (4 * nfull < nv) {
      const bool in = 4 * nfull + g < nv;
      const double x = in ? ca[4 * nfull] : 0.0, y = in ? cb[4 * nfull] : 0.0;
      a1 = __builtin_amdgcn_mfma_f64_16x16x4f64(x, y, a1, 0, 0, 0);
    }
    a0 += a1;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int r = 16 * bi + 4 * s + g, c = 16 * bj + mr;
      if (r <= c && c < n) {
        Pm[(size_t)r * n + c] = 2.0 * a0[s];
        Pm[(size_t)c * n + r] = 2.0 * a0[s];
      }
    }
  }
}

}  // namespace

extern "C" long long pyseqm_eigh_density_workspace(int nact, int nmax) {
  if (nact < 0 || nmax < 0) return -1;
  return 4LL * nact * nmax * nmax;
}

// waves per workgroup and register slots per thread: the 4 NW x 16 thread grid covers 48, 96 or 192
// orbitals.  The smaller two take 310 to 320 registers, one wave per SIMD; with more blocks than run so
// at once they are held to 256, for two (some 30 spilled).  Blocks (us, one wave -> two): 4096 x 8 173 -> 126,
// 4096 x 20 278 -> 198, 1024 x 50 402 -> 278, 512 x 96 414 -> 291; 1024 x 14 82 -> 88, 256 x 50 133 -> 132, and the
// eigenpairs of 32 clusters of 3-12 waters 2 % slower: above the number of blocks that fills 256 CUs.
template <int NW, int RR, int RC, bool EVEC>
void launch_eigh_grid(const pyseqm_layout_t* L, const int* idx, int nact, int nmax, const double* F, double* out,
                      double* ws, int* fail, const long long* orb_off, double* evals, size_t lds, hipStream_t s) {
  if (nact <= 4 / NW * 256)
    k_eigh_density<NW, RR, RC, EVEC, false, 1><<<nact, 64 * NW, lds, s>>>(*L, idx, F, out, ws, nmax, fail, orb_off,
                                                                         evals, nullptr);
  else
    k_eigh_density<NW, RR, RC, EVEC, false, 2><<<nact, 64 * NW, lds, s>>>(*L, idx, F, out, ws, nmax, fail, orb_off,
                                                                         evals, nullptr);
}
template <bool EVEC>
void launch_eigh(const pyseqm_layout_t* L, const int* idx, int nact, int nmax, const double* F, double* out,
                 double* ws, int* fail, const long long* orb_off, double* evals, size_t lds, hipStream_t s) {
  if (nmax <= 48)
    launch_eigh_grid<1, 12, 3, EVEC>(L, idx, nact, nmax, F, out, ws, fail, orb_off, evals, lds, s);
  else if (nmax <= 96)
    launch_eigh_grid<4, 6, 6, EVEC>(L, idx, nact, nmax, F, out, ws, fail, orb_off, evals, lds, s);
  else
    k_eigh_density<8, 6, 12, EVEC, false, 2><<<nact, 512, lds, s>>>(*L, idx, F, out, ws, nmax, fail, orb_off, evals,
                                                                   nullptr);
}

extern "C" int pyseqm_eigh_density_lds_ok(int norb, int nocc) {
  if (norb < 1 || norb > kEighMaxN || nocc < 0 || nocc > norb) return 0;
  return rule_doubles(norb, nocc) <= kLdsDoubles;
}

extern "C" int pyseqm_eigh_density(const pyseqm_layout_t* L, const int* idx, int nact, int nmax, int nocc_max,
                                   const double* F, double* P, double* ws, int* fail, void* stream) {
  if (!L || nact < 0 || nmax < 1 || nmax > kEighMaxN || nocc_max < 0 || nocc_max > nmax || !fail)
    return PYSEQM_EINVAL;
  if (!pyseqm_eigh_density_lds_ok(nmax, nocc_max)) return PYSEQM_EINVAL;
  if (nact == 0) return PYSEQM_OK;
  const size_t lds = (size_t)lds_doubles(nmax, nocc_max) * sizeof(double);
  hipStream_t s = (hipStream_t)stream;
  launch_eigh<false>(L, idx, nact, nmax, F, P, ws, fail, nullptr, nullptr, lds, s);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}

extern "C" int pyseqm_eigh_density_large(const pyseqm_layout_t* L, const int* idx, int nact, int nmax,
                                         const double* F, double* P, double* ws, double* Z, int* fail,
                                         void* stream) {
  if (!L || nact < 0 || nmax < 1 || nmax > kEighMaxN || !fail || !Z) return PYSEQM_EINVAL;
  if (nact == 0) return PYSEQM_OK;
  if (nmax <= 48) {  // any occupation fits LDS; the 192-row variant's panel factors would not fit a slot below 32
    launch_eigh<false>(L, idx, nact, nmax, F, P, ws, fail, nullptr, nullptr, lds_doubles(nmax, nmax) * sizeof(double),
                       (hipStream_t)stream);
    return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
  }
  static_assert(3 * 49 * 49 >= 12 * kTPanel, "the panel factors lie behind the reflectors in a molecule's slot");
  const size_t lds = (size_t)(zregion(0, 0, 192) + 6 * nmax + kLdsExtra) * sizeof(double);
  k_eigh_density<8, 6, 12, false, true, 2>
      <<<nact, 512, lds, (hipStream_t)stream>>>(*L, idx, F, P, ws, nmax, fail, nullptr, nullptr, Z);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}

extern "C" int pyseqm_eigh_vectors(const pyseqm_layout_t* L, const int* idx, int nact, int nmax, const double* F,
                                   const long long* orb_off, double* evals, double* Q, double* ws, int* fail,
                                   void* stream) {
  if (!L || nact < 0 || nmax < 1 || nmax > kEighMaxN || !fail || !orb_off || !evals) return PYSEQM_EINVAL;
  if (nact == 0) return PYSEQM_OK;
  if (!pyseqm_eigh_density_lds_ok(nmax, nmax)) {  // above 139 orbitals: vectors in Q
    const size_t lds = (size_t)(zregion(0, 0, 192) + 6 * nmax + kLdsExtra) * sizeof(double);
    k_eigh_density<8, 6, 12, true, true, 2>
        <<<nact, 512, lds, (hipStream_t)stream>>>(*L, idx, F, Q, ws, nmax, fail, orb_off, evals, nullptr);
    return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
  }
  const size_t lds = (size_t)lds_doubles(nmax, nmax) * sizeof(double);
  launch_eigh<true>(L, idx, nact, nmax, F, Q, ws, fail, orb_off, evals, lds, (hipStream_t)stream);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}
