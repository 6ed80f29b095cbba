// Thermal (Fermi) density and the Krylov-subspace (KSA) XL-BOMD kernel on the packed batch.
//
//   * Fermi occupations f = 1 / (1 + exp((e - mu) / kT)) of every eigenpair, the chemical potential
//     by Newton steps from the HOMO/LUMO midpoint with the reference's batch-wide stop, the density
//     D = 2 Q diag(f) Q^T and the entropy (fermi_q.py:8-72).
//   * FP64 products of n x n blocks (C = op(A) op(B)) for the eigenbasis transforms of the
//     canonical density-matrix perturbation theory, its recursion in the eigenbasis and the
//     chemical-potential shift (canon_dm_prt.py:6-39).
//   * Per-molecule Frobenius products, block updates and small dense solves of the rank-m
//     Krylov fit (seqm/dynamics/xlbomd.py:243-339).
// Every block is a molecule's packed n x n matrix at mol_mat_off; eigenvalues and occupations
// are at orb_off[m] + j.  Reductions run in a fixed order: reruns are bitwise identical.
#include "common.h"

using namespace pyseqm;

typedef double doublex4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int kFermiIter = 64;      // fermi_q.py:12
constexpr double kOccTol = 1.0e-9;  // fermi_q.py:14 (float64)
constexpr double kEntEps = 1.0e-14;
constexpr double kTiny = 1.0e-30;
constexpr int kMaxRank = 8;         // largest Krylov rank of pyseqm_small_solve

__device__ inline double sigm(double x) { return 1.0 / (1.0 + exp(-x)); }

// fixed-order sum over a 256-thread block; every thread gets the total
__device__ inline double block_sum256(double v, double* red) {
  v = wave_sum(v);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// Newton steps for mu, one wave per molecule: every step's mu and whether |nocc - sum f| <= tol
// are recorded (the batch stops at the first step at which every molecule is converged).  A step depends on
// mu alone, so once a mu returns (the last one, or the one before it: rounding can leave a pair) the rest of
// the record repeats and is filled in: 43 us with all 64 steps taken, 14 here for 32 clusters of 3-12 waters.
__global__ __launch_bounds__(64) void k_fermi_newton(pyseqm_layout_t L, const int* __restrict__ idx,
                                                     const long long* __restrict__ orb_off,
                                                     const double* __restrict__ evals, double beta,
                                                     double* __restrict__ mu_hist, unsigned char* __restrict__ conv) {
  const int slot = blockIdx.x, lane = threadIdx.x;
  const int m = idx[slot];
  const int n = L.mol_norb[m], N = L.mol_nocc[m];
  const double* e = evals + orb_off[m];
  double mu = 0.5 * (e[N - 1] + e[N]), mu1 = 0.0;  // mu1: of the step before
  bool c1 = false;
  for (int t = 0; t < kFermiIter; ++t) {
    double occ = 0.0, docc = 0.0;
    for (int i = lane; i < n; i += 64) {
      const double f = sigm(-beta * (e[i] - mu));
      occ += f;
      docc += beta * f * (1.0 - f);
    }
    occ = wave_sum(occ);
    docc = fmax(wave_sum(docc), kTiny);
    const bool ct = fabs((double)N - occ) <= kOccTol;
    if (lane == 0) {
      mu_hist[(size_t)slot * kFermiIter + t] = mu;
      conv[(size_t)slot * kFermiIter + t] = ct;
    }
    const double next = mu + ((double)N - occ) / docc;
    const bool same = next == mu;
    if (same || (t > 0 && next == mu1)) {  // uniform: the sums are the same in every lane
      for (int u = t + 1 + lane; u < kFermiIter; u += 64) {
        const bool now = same || ((u - t) & 1) == 0;  // this step's mu again, or that of the step before
        mu_hist[(size_t)slot * kFermiIter + u] = now ? mu : mu1;
        conv[(size_t)slot * kFermiIter + u] = now ? ct : c1;
      }
      break;
    }
    mu1 = mu;
    c1 = ct;
    mu = next;
  }
}

// The first step at which every listed molecule is converged (the last step if none is).
__global__ __launch_bounds__(256) void k_fermi_pick(int nact, const unsigned char* __restrict__ conv,
                                                    int* __restrict__ kout) {
  int K = kFermiIter - 1;
  for (int t = 0; t < kFermiIter; ++t) {
    int all = 1;
    for (int s = threadIdx.x; s < nact; s += blockDim.x) all &= conv[(size_t)s * kFermiIter + t];
    if (__syncthreads_and(all)) {
      K = t;
      break;
    }
  }
  if (threadIdx.x == 0) *kout = K;
}

// Occupations and entropy at the chosen step's mu, one block per molecule.
__global__ __launch_bounds__(256) void k_fermi_occ(pyseqm_layout_t L, const int* __restrict__ idx,
                                                   const long long* __restrict__ orb_off,
                                                   const double* __restrict__ evals, double beta, double kB,
                                                   const double* __restrict__ mu_hist,
                                                   const int* __restrict__ kpick, double* __restrict__ occ,
                                                   double* __restrict__ mu_out, double* __restrict__ S) {
  __shared__ double red[4];
  const int slot = blockIdx.x, tid = threadIdx.x;
  const int m = idx[slot];
  const int n = L.mol_norb[m];
  const double mu = mu_hist[(size_t)slot * kFermiIter + *kpick];
  const double* e = evals + orb_off[m];
  double s = 0.0;
  for (int i = tid; i < n; i += 256) {
    const double fi = sigm(-beta * (e[i] - mu));
    occ[orb_off[m] + i] = fi;
    if (fi > kEntEps && 1.0 - fi > kEntEps) s += -kB * (fi * log(fi) + (1.0 - fi) * log(1.0 - fi));
  }
  s = block_sum256(s, red);
  if (tid == 0) {
    S[m] = s;
    mu_out[m] = mu;
  }
}

// D = 2 Q diag(f) Q^T: a 16 x 16 tile of the upper triangle per wave on FP64 MFMA, both operands rows of Q as
// they lie in memory (a tile's rows are shared by its neighbours through the L2); elements r <= c go to
// both triangles.  A block per molecule with one element per thread took 66 us for 32 clusters of 3-12
// waters, this and k_fermi_occ 10.
__global__ __launch_bounds__(256) void k_fermi_density(pyseqm_layout_t L, const int* __restrict__ idx,
                                                       const long long* __restrict__ orb_off,
                                                       const double* __restrict__ occ,
                                                       const double* __restrict__ Q, double* __restrict__ D) {
  const int m = idx[blockIdx.y];
  const int n = L.mol_norb[m];
  const int nt = (n + 15) / 16;
  int rem = blockIdx.x * 4 + (threadIdx.x >> 6), bi = 0;
  if (rem >= nt * (nt + 1) / 2) return;
  while (rem >= nt - bi) {
    rem -= nt - bi;
    ++bi;
  }
  const int bj = bi + rem, mr = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
  const size_t mo = L.mol_mat_off[m];
  const double* f = occ + orb_off[m];
  const double* ca = Q + mo + (size_t)min(16 * bi + mr, n - 1) * n;
  const double* cb = Q + mo + (size_t)min(16 * bj + mr, n - 1) * n;
  doublex4 acc = {0.0, 0.0, 0.0, 0.0};
  int k0 = 0;
  for (; k0 + 16 <= n; k0 += 16) {  // the loads of four steps first
    double x[4], y[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      x[q] = ca[k0 + 4 * q + g] * f[k0 + 4 * q + g];
      y[q] = cb[k0 + 4 * q + g];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x[q], y[q], acc, 0, 0, 0);
  }
  for (; k0 < n; k0 += 4) {
    const int k = min(k0 + g, n - 1);
    const double a = k0 + g < n ? ca[k] * f[k] : 0.0;
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, cb[k], acc, 0, 0, 0);
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int r = 16 * bi + 4 * s + g, c = 16 * bj + mr;
    if (r <= c && c < n) {
      D[mo + (size_t)r * n + c] = 2.0 * acc[s];
      D[mo + (size_t)c * n + r] = 2.0 * acc[s];
    }
  }
}

// C = op(A) op(B) per listed molecule, 16 x 16 output tiles through LDS.
template <bool TA, bool TB>
__global__ __launch_bounds__(256) void k_block_gemm(pyseqm_layout_t L, const int* __restrict__ idx,
                                                    const double* __restrict__ A, const double* __restrict__ B,
                                                    double* __restrict__ C) {
  __shared__ double As[16][17], Bs[16][17];
  const int m = idx[blockIdx.y];
  const int n = L.mol_norb[m];
  const int nt = (n + 15) / 16;
  if ((int)blockIdx.x >= nt * nt) return;  // uniform over the block
  const int ti = blockIdx.x / nt, tj = blockIdx.x - (blockIdx.x / nt) * nt;
  const int ty = threadIdx.x >> 4, tx = threadIdx.x & 15;
  const size_t mo = L.mol_mat_off[m];
  const double* Am = A + mo;
  const double* Bm = B + mo;
  const int r = ti * 16 + ty, c = tj * 16 + tx;
  double acc = 0.0;
  for (int k0 = 0; k0 < n; k0 += 16) {
    const int ka = k0 + tx, kb = k0 + ty;
    As[ty][tx] = (r < n && ka < n) ? (TA ? Am[(size_t)ka * n + r] : Am[(size_t)r * n + ka]) : 0.0;
    Bs[ty][tx] = (kb < n && c < n) ? (TB ? Bm[(size_t)c * n + kb] : Bm[(size_t)kb * n + c]) : 0.0;
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) acc += As[ty][kk] * Bs[kk][tx];
    __syncthreads();
  }
  if (r < n && c < n) C[mo + (size_t)r * n + c] = acc;
}

// Recursive Fermi-operator expansion of the perturbation in the eigenbasis, element by element:
// p0 = 1/2 - 2^(-2-m) beta (e - mu), P1 = -2^(-2-m) beta Y, then m steps of
// dX1 = p0_i P1 + P1 p0_j, p0 <- p0^2 / (2 (p0^2 - p0) + 1), P1 <- (dX1 + 2 (P1 - dX1) p0_j) / (2 (p0_i^2 - p0_i) + 1).
__global__ __launch_bounds__(256) void k_canon_elem(pyseqm_layout_t L, const int* __restrict__ idx,
                                                    const long long* __restrict__ orb_off,
                                                    const double* __restrict__ evals, const double* __restrict__ mu,
                                                    double beta, int steps, double* __restrict__ Y) {
  const int m = idx[blockIdx.y];
  const int n = L.mol_norb[m];
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= n * n) return;
  const int i = t / n, j = t - (t / n) * n;
  const double* e = evals + orb_off[m];
  const double cn = ldexp(beta, -2 - steps);
  double p0i = 0.5 - cn * (e[i] - mu[m]);
  double p0j = 0.5 - cn * (e[j] - mu[m]);
  double* y = Y + L.mol_mat_off[m] + t;
  double P1 = -cn * *y;
  for (int s = 0; s < steps; ++s) {
    const double p02i = p0i * p0i, p02j = p0j * p0j;
    const double dX1 = p0i * P1 + P1 * p0j;
    const double iDi = 1.0 / (2.0 * (p02i - p0i) + 1.0);
    const double iDj = 1.0 / (2.0 * (p02j - p0j) + 1.0);
    p0i = iDi * p02i;
    p0j = iDj * p02j;
    P1 = iDi * (dX1 + 2.0 * (P1 - dX1) * p0j);
  }
  *y = P1;
}

// First-order response of the closed-shell density D = 2 sum_occ c c^T to a symmetric Fock
// perturbation, in the eigenbasis: dD'_ia = dD'_ai = 2 F'_ia / (e_i - e_a) for i occupied and a
// virtual (the nocc lowest eigenpairs), zero in the occupied-occupied and virtual-virtual blocks.
// The operator is self-adjoint, so it is also the transpose the SCF implicit backward applies
// (the eigh backward of sym_eig_trunc1 inside scf_loop.py:1779-1993).
__global__ __launch_bounds__(256) void k_response_elem(pyseqm_layout_t L, const int* __restrict__ idx,
                                                       const long long* __restrict__ orb_off,
                                                       const double* __restrict__ evals, double* __restrict__ Y) {
  const int m = idx[blockIdx.y];
  const int n = L.mol_norb[m];
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= n * n) return;
  const int i = t / n, j = t - (t / n) * n;
  const int nocc = L.mol_nocc[m];
  const double* e = evals + orb_off[m];
  double* y = Y + L.mol_mat_off[m] + t;
  const bool oi = i < nocc, oj = j < nocc;
  *y = oi == oj ? 0.0 : *y * 2.0 / (oi ? e[i] - e[j] : e[j] - e[i]);
}

// The chemical-potential shift that keeps the trace: P1 += diag(dp/dmu) dmu1,
// dmu1 = -tr P1 / sum dp/dmu, dp/dmu = beta p0 (1 - p0) of the final p0; one block per molecule.
__global__ __launch_bounds__(256) void k_canon_shift(pyseqm_layout_t L, const int* __restrict__ idx,
                                                     const long long* __restrict__ orb_off,
                                                     const double* __restrict__ evals, const double* __restrict__ mu,
                                                     double beta, int steps, double* __restrict__ Y) {
  __shared__ double red[4];
  __shared__ double dp[256];
  const int m = idx[blockIdx.x], tid = threadIdx.x;
  const int n = L.mol_norb[m];
  double* Ym = Y + L.mol_mat_off[m];
  const double* e = evals + orb_off[m];
  const double cn = ldexp(beta, -2 - steps);
  double tr = 0.0, sdp = 0.0;
  for (int i = tid; i < n; i += 256) {
    double p0 = 0.5 - cn * (e[i] - mu[m]);
    for (int s = 0; s < steps; ++s) {
      const double p02 = p0 * p0;
      p0 = p02 / (2.0 * (p02 - p0) + 1.0) ;
    }
    dp[i] = beta * p0 * (1.0 - p0);
    tr += Ym[(size_t)i * n + i];
    sdp += dp[i];
  }
  tr = block_sum256(tr, red);
  sdp = block_sum256(sdp, red);
  const double dmu1 = -tr / sdp;
  for (int i = tid; i < n; i += 256) Ym[(size_t)i * n + i] += dp[i] * dmu1;
}

// out[slot] = sum over the block of A * B (Frobenius product), one block per molecule
__global__ __launch_bounds__(256) void k_block_dot(pyseqm_layout_t L, const int* __restrict__ idx,
                                                   const double* __restrict__ A, const double* __restrict__ B,
                                                   double* __restrict__ out) {
  __shared__ double red[4];
  const int m = idx[blockIdx.x];
  const int n = L.mol_norb[m];
  const size_t mo = L.mol_mat_off[m];
  double s = 0.0;
  for (int t = threadIdx.x; t < n * n; t += 256) s += A[mo + t] * B[mo + t];
  s = block_sum256(s, red);
  if (threadIdx.x == 0) out[m] = s;
}

// Y <- Y + s c_m X (mode 0), Y / sqrt(c_m) (1), s (Y - X) (2), s c_m X (3), Y + s X (4);
// c_m = c[m * cstride].
__global__ __launch_bounds__(256) void k_block_axpy(pyseqm_layout_t L, const int* __restrict__ idx, int mode,
                                                    double s, const double* __restrict__ c, int cstride,
                                                    const double* __restrict__ X, double* __restrict__ Y) {
  const int m = idx[blockIdx.y];
  const int n = L.mol_norb[m];
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= n * n) return;
  const size_t o = L.mol_mat_off[m] + t;
  const double cm = c ? c[(size_t)m * cstride] : 0.0;
  switch (mode) {
    case 0: Y[o] += s * cm * X[o]; break;
    case 1: Y[o] /= sqrt(cm); break;
    case 2: Y[o] = s * (Y[o] - X[o]); break;
    case 3: Y[o] = s * cm * X[o]; break;
    default: Y[o] += s * X[o]; break;
  }
}

// a[i][r] <- the solution of a[0 .. r-1][0 .. r-1] x = a[0 .. r-1][r] (Gaussian elimination with partial pivoting,
// r <= kMaxRank), one thread.
typedef double FitSystem[kMaxRank][kMaxRank + 1];
__device__ inline void eliminate(FitSystem& a, int r) {
  for (int k = 0; k < r; ++k) {
    int p = k;
    for (int i = k + 1; i < r; ++i)
      if (fabs(a[i][k]) > fabs(a[p][k])) p = i;
    if (p != k)
      for (int j = k; j <= r; ++j) {
        const double t = a[k][j];
        a[k][j] = a[p][j];
        a[p][j] = t;
      }
    for (int i = k + 1; i < r; ++i) {
      const double l = a[i][k] / a[k][k];
      for (int j = k; j <= r; ++j) a[i][j] -= l * a[k][j];
    }
  }
  for (int i = r - 1; i >= 0; --i) {
    double v = a[i][r];
    for (int j = i + 1; j < r; ++j) v -= a[i][j] * a[j][r];
    a[i][r] = v / a[i][i];
  }
}

// alpha = O^{-1} rhs per molecule; O[m][i][j] at m * kMaxRank^2 + i * kMaxRank + j, rhs / alpha at
// m * kMaxRank + i.
__global__ __launch_bounds__(64) void k_small_solve(const int* __restrict__ idx, int nact, int r,
                                                    const double* __restrict__ O, const double* __restrict__ rhs,
                                                    double* __restrict__ alpha) {
  const int s = blockIdx.x * 64 + threadIdx.x;
  if (s >= nact) return;
  const int m = idx[s];
  FitSystem a;
  for (int i = 0; i < r; ++i) {
    for (int j = 0; j < r; ++j) a[i][j] = O[(size_t)m * kMaxRank * kMaxRank + i * kMaxRank + j];
    a[i][r] = rhs[(size_t)m * kMaxRank + i];
  }
  eliminate(a, r);
  for (int i = 0; i < r; ++i) alpha[(size_t)m * kMaxRank + i] = a[i][r];
}

// ------------------------------------------------------------------ Krylov step
// One workgroup per molecule carries a Krylov vector from its residual to the fit, with only the Fock build
// G(V_k) between k_krylov_start and k_krylov_response: the Frobenius products are sums over one block, so a
// launch each (26 a step at rank 3, 5.8 us each, and as many updates and copies) bought nothing.
constexpr int kKrylovThreads = 1024, kKrylovWaves = kKrylovThreads / 64;

// fixed-order sums of q values over the workgroup; every thread gets them.  red[i][kKrylovWaves] takes the total:
// one thread per value adds the waves (every thread adding them all is 8 q LDS reads in each wave)
template <int NQ>
__device__ inline void block_sums(double (&v)[NQ], int q, double (*red)[kKrylovWaves + 1]) {
  const int w = threadIdx.x >> 6;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NQ; ++i)
    if (i < q) {
      const double s = wave_sum(v[i]);
      if ((threadIdx.x & 63) == 0) red[i][w] = s;
    }
  __syncthreads();
  if ((int)threadIdx.x < q) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < kKrylovWaves; ++k) s += red[threadIdx.x][k];
    red[threadIdx.x][kKrylovWaves] = s;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NQ; ++i)
    if (i < q) v[i] = red[i][kKrylovWaves];
}

// V_k = the residual (k = 0: D - P, kept as dDS; else W_{k-1}), modified Gram-Schmidt against V_0 .. V_{k-1}
// in the Frobenius product, normalised.  A thread keeps to its own elements throughout.
__global__ __launch_bounds__(kKrylovThreads) void k_krylov_start(pyseqm_layout_t L, const int* __restrict__ idx,
                                                                int k, const double* __restrict__ D,
                                                                const double* __restrict__ P,
                                                                double* __restrict__ dDS, double* __restrict__ V,
                                                                const double* __restrict__ W, size_t stride) {
  __shared__ double red[1][kKrylovWaves + 1];
  const int m = idx[blockIdx.x];
  const int n = L.mol_norb[m], n2 = n * n;
  const size_t mo = L.mol_mat_off[m];
  double* v = V + k * stride + mo;
  double s[1] = {0.0};
  constexpr int kU = 8;  // loads in flight per thread and operand
  const double* a0 = k == 0 ? D + mo : W + (k - 1) * stride + mo;
  const double* b0 = k == 0 ? P + mo : V + mo;
  for (int t0 = threadIdx.x; t0 < n2; t0 += kU * kKrylovThreads) {
    double a[kU], b[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int t = min(t0 + u * kKrylovThreads, n2 - 1);
      a[u] = a0[t];
      b[u] = b0[t];
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int t = t0 + u * kKrylovThreads;
      if (t >= n2) continue;
      const double x = k == 0 ? a[u] - b[u] : a[u];
      if (k == 0) dDS[mo + t] = x;
      s[0] += x * (k == 0 ? x : b[u]);
      v[t] = x;
    }
  }
  block_sums(s, 1, red);
  for (int j = 0; j < k; ++j) {
    const double c = -s[0];
    const double* vj = V + j * stride + mo;
    const bool last = j + 1 == k;  // <V_k, V_{j+1}> for the next vector, at last <V_k, V_k>
    const double* vn = V + (last ? j : j + 1) * stride + mo;
    s[0] = 0.0;
    for (int t0 = threadIdx.x; t0 < n2; t0 += kU * kKrylovThreads) {
      double a[kU], b[kU], d[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int t = min(t0 + u * kKrylovThreads, n2 - 1);
        a[u] = t0 + u * kKrylovThreads < n2 ? v[t] : 0.0;  // its own elements only
        b[u] = vj[t];
        d[u] = vn[t];
      }
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int t = t0 + u * kKrylovThreads;
        if (t >= n2) continue;
        const double x = a[u] + c * b[u];
        v[t] = x;
        s[0] += x * (last ? x : d[u]);
      }
    }
    block_sums(s, 1, red);
  }
  const double nrm = sqrt(s[0]);
#pragma unroll 4
  for (int t = threadIdx.x; t < n2; t += kKrylovThreads) v[t] /= nrm;
}

// The fit's system of the k earlier vectors into LDS (early in a kernel: the reads take their time), and with
// row k from q[i] = <W_k, W_i> (i <= k) and q[k + 1] = <W_k, dDS> its solution; thread 0.  In LDS, not in
// registers: indexed by pivots it would go to scratch memory.
__device__ inline void krylov_fetch(int m, int k, const double* O, const double* rhs, FitSystem& a) {
  const int i = threadIdx.x / (kMaxRank + 1), j = threadIdx.x % (kMaxRank + 1);
  if (i < k && j < k) a[i][j] = O[(size_t)m * kMaxRank * kMaxRank + i * kMaxRank + j];
  if (i < k && j == k + 1) a[i][j] = rhs[(size_t)m * kMaxRank + i];
}
__device__ inline void krylov_solve(int m, int k, const double (&q)[kMaxRank + 1], double* O, double* rhs,
                                    double* alpha, FitSystem& a) {
  double* Om = O + (size_t)m * kMaxRank * kMaxRank;
#pragma unroll
  for (int i = 0; i <= kMaxRank; ++i) {
    if (i <= k) {
      Om[k * kMaxRank + i] = Om[i * kMaxRank + k] = q[i];
      a[k][i] = a[i][k] = q[i];
    } else if (i == k + 1) {
      rhs[(size_t)m * kMaxRank + k] = a[k][k + 1] = q[i];
    }
  }
  eliminate(a, k + 1);
  for (int i = 0; i <= k; ++i) alpha[(size_t)m * kMaxRank + i] = a[i][k + 1];
}

// W_k <- W_k - V_k, the fit's row and its solution, where W_k holds the response of V_k
__global__ __launch_bounds__(kKrylovThreads) void k_krylov_fit(pyseqm_layout_t L, const int* __restrict__ idx, int k,
                                                              const double* __restrict__ V, double* __restrict__ W,
                                                              size_t stride, const double* __restrict__ dDS,
                                                              double* __restrict__ O, double* __restrict__ rhs,
                                                              double* __restrict__ alpha) {
  __shared__ double red[kMaxRank + 1][kKrylovWaves + 1];
  __shared__ FitSystem fit;
  const int m = idx[blockIdx.x];
  const int n = L.mol_norb[m], n2 = n * n;
  const size_t mo = L.mol_mat_off[m];
  krylov_fetch(m, k, O, rhs, fit);
  double q[kMaxRank + 1];
#pragma unroll
  for (int i = 0; i <= kMaxRank; ++i) q[i] = 0.0;
  for (int t = threadIdx.x; t < n2; t += kKrylovThreads) {
    const size_t o = mo + t;
    const double w = W[k * stride + o] - V[k * stride + o];
    W[k * stride + o] = w;
#pragma unroll
    for (int i = 0; i <= kMaxRank; ++i)
      if (i <= k + 1) q[i] += w * (i < k ? W[i * stride + o] : (i == k ? w : dDS[o]));
  }
  block_sums(q, k + 2, red);
  if (threadIdx.x == 0) krylov_solve(m, k, q, O, rhs, alpha, fit);
}

// Doubles of LDS of k_krylov_response: Q and two more blocks, the recursion's tables, the shift's weights
__host__ __device__ inline int krylov_ld(int n) { return n | 1; }
inline long long krylov_lds(int n, int steps) { return 3LL * n * krylov_ld(n) + (2LL * steps + 2) * n; }

// One 16 x 16 tile of sum_k a(row, k) b(k, column) at rows r0, columns c0 (FP64 MFMA; operands outside the block are
// read at its edge: those elements are not used)
template <class A, class B>
__device__ inline doublex4 block_tile(int n, int r0, int c0, A a, B b) {
  const int mr = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
  const int r = min(r0 + mr, n - 1), c = min(c0 + mr, n - 1);
  doublex4 acc = {0.0, 0.0, 0.0, 0.0};
  int k0 = 0;
  for (; k0 + 16 <= n; k0 += 16) {  // the reads of four steps first
    double x[4], y[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      x[q] = a(r, k0 + 4 * q + g);
      y[q] = b(k0 + 4 * q + g, c);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x[q], y[q], acc, 0, 0, 0);
  }
  for (; k0 < n; k0 += 4) {
    const int kk = min(k0 + g, n - 1);
    const double x = a(r, kk);
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(k0 + g < n ? x : 0.0, b(kk, c), acc, 0, 0, 0);
  }
  return acc;
}

// The whole response of V_k in one launch, blocks of which three fit LDS: W_k = Q canon(Q^T G Q) Q^T - V_k
// (k_canon_elem, k_canon_shift), then the fit as in k_krylov_fit.  Four products on FP64 MFMA, a 16 x 16
// tile per wave at a time; the recursion's p0 and 1 / (2 (p0^2 - p0) + 1) of every step are formed once per
// orbital instead of per element (two divisions a step each).  What bounds it: the chain of four products and
// their barriers in one workgroup, and the fetch of its instructions (a form with every tile of a wave
// unrolled in registers, two blocks in LDS, took 42 us).  32 clusters of 3-12 waters: four block products,
// recursion and shift took 40 us per vector, the products of the fit and their updates 40; now 38.
__global__ __launch_bounds__(kKrylovThreads) void k_krylov_response(
    pyseqm_layout_t L, const int* __restrict__ idx, const long long* __restrict__ orb_off,
    const double* __restrict__ evals, const double* __restrict__ mu, double beta, int steps,
    const double* __restrict__ Q, const double* __restrict__ G, int k, const double* __restrict__ V, double* W,
    size_t stride, const double* __restrict__ dDS, double* __restrict__ O, double* __restrict__ rhs,
    double* __restrict__ alpha) {
  extern __shared__ __align__(16) double lds[];
  __shared__ double red[kMaxRank + 1][kKrylovWaves + 1];
  __shared__ FitSystem fit;
  const int m = idx[blockIdx.x];
  const int n = L.mol_norb[m], ld = krylov_ld(n), nt = (n + 15) / 16;
  const size_t mo = L.mol_mat_off[m];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, mr = lane & 15, g = lane >> 4;
  double* Qs = lds;
  double* As = Qs + n * ld;
  double* Bs = As + n * ld;
  double* p0s = Bs + n * ld;              // [steps + 1][n]
  double* iDs = p0s + (steps + 1) * n;    // [steps][n]
  double* dp = iDs + steps * n;
  const double cn = ldexp(beta, -2 - steps);
  krylov_fetch(m, k, O, rhs, fit);
  for (int t0 = tid; t0 < n * n; t0 += 4 * kKrylovThreads) {  // Q and G, eight loads in flight per thread
    double a[4], b[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const size_t o = mo + min(t0 + q * kKrylovThreads, n * n - 1);
      a[q] = Q[o];
      b[q] = G[o];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int t = t0 + q * kKrylovThreads, r = t / n;
      if (t < n * n) {
        Qs[r * ld + t - r * n] = a[q];
        As[r * ld + t - r * n] = b[q];
      }
    }
  }
  double sums[kMaxRank + 1];
#pragma unroll
  for (int i = 0; i <= kMaxRank; ++i) sums[i] = 0.0;
  for (int i = tid; i < n; i += kKrylovThreads) {
    double p = 0.5 - cn * (evals[orb_off[m] + i] - mu[m]);
    p0s[i] = p;
    for (int s = 0; s < steps; ++s) {
      const double p2 = p * p, d = 1.0 / (2.0 * (p2 - p) + 1.0);
      p = d * p2;
      iDs[s * n + i] = d;
      p0s[(s + 1) * n + i] = p;
    }
    dp[i] = beta * p * (1.0 - p);
    sums[1] += dp[i];
  }
  __syncthreads();
  for (int t = wave; t < nt * nt; t += kKrylovWaves) {  // B = G Q
    const int r0 = 16 * (t / nt), c0 = 16 * (t % nt), j = c0 + mr;
    const doublex4 x = block_tile(n, r0, c0, [&](int r, int kk) { return As[r * ld + kk]; },
                                  [&](int kk, int c) { return Qs[kk * ld + c]; });
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (r0 + 4 * q + g < n && j < n) Bs[(r0 + 4 * q + g) * ld + j] = x[q];
  }
  __syncthreads();
  for (int t = wave; t < nt * nt; t += kKrylovWaves) {  // A = the recursion on Q^T B
    const int r0 = 16 * (t / nt), c0 = 16 * (t % nt), j = min(c0 + mr, n - 1);
    doublex4 x = block_tile(n, r0, c0, [&](int r, int kk) { return Qs[kk * ld + r]; },
                            [&](int kk, int c) { return Bs[kk * ld + c]; });
    int i[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      i[q] = min(r0 + 4 * q + g, n - 1);
      x[q] *= -cn;
    }
    double pj = p0s[j];
    for (int s = 0; s < steps; ++s) {
      const double pn = p0s[(s + 1) * n + j];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const double dX1 = p0s[s * n + i[q]] * x[q] + x[q] * pj;
        x[q] = iDs[s * n + i[q]] * (dX1 + 2.0 * (x[q] - dX1) * pn);
      }
      pj = pn;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (r0 + 4 * q + g < n && c0 + mr < n) {
        As[i[q] * ld + j] = x[q];
        if (i[q] == j) sums[0] += x[q];
      }
  }
  block_sums(sums, 2, red);
  const double dmu1 = -sums[0] / sums[1];
  for (int i = tid; i < n; i += kKrylovThreads) As[i * ld + i] += dp[i] * dmu1;
  __syncthreads();
  for (int t = wave; t < nt * nt; t += kKrylovWaves) {  // B = Q A
    const int r0 = 16 * (t / nt), c0 = 16 * (t % nt), j = c0 + mr;
    const doublex4 x = block_tile(n, r0, c0, [&](int r, int kk) { return Qs[r * ld + kk]; },
                                  [&](int kk, int c) { return As[kk * ld + c]; });
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (r0 + 4 * q + g < n && j < n) Bs[(r0 + 4 * q + g) * ld + j] = x[q];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i <= kMaxRank; ++i) sums[i] = 0.0;
  for (int t = wave; t < nt * nt; t += kKrylovWaves) {  // W_k = B Q^T - V_k and its products with the others
    const int r0 = 16 * (t / nt), c0 = 16 * (t % nt);
    size_t o[4];
    bool in[4];
    double v[4], d[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {  // loads first, at edge addresses outside the block
      const int i = r0 + 4 * q + g, j = c0 + mr;
      in[q] = i < n && j < n;
      o[q] = mo + (size_t)min(i, n - 1) * n + min(j, n - 1);
      v[q] = V[k * stride + o[q]];
      d[q] = dDS[o[q]];
    }
    doublex4 x = block_tile(n, r0, c0, [&](int r, int kk) { return Bs[r * ld + kk]; },
                            [&](int kk, int c) { return Qs[c * ld + kk]; });
    double wd = 0.0, ww = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      x[q] = in[q] ? x[q] - v[q] : 0.0;
      wd += x[q] * (in[q] ? d[q] : 0.0);
      ww += x[q] * x[q];
    }
#pragma unroll
    for (int p = 0; p < kMaxRank; ++p)
      if (p < k) {
#pragma unroll
        for (int q = 0; q < 4; ++q) sums[p] += x[q] * (in[q] ? W[p * stride + o[q]] : 0.0);
      } else if (p == k) {
        sums[p] += ww;
        sums[p + 1] += wd;
      }
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (in[q]) W[k * stride + o[q]] = x[q];
  }
  block_sums(sums, k + 2, red);
  if (tid == 0) krylov_solve(m, k, sums, O, rhs, alpha, fit);
}

// out = -sum_r alpha_r V_r
__global__ __launch_bounds__(256) void k_krylov_combine(pyseqm_layout_t L, const int* __restrict__ idx, int r,
                                                        const double* __restrict__ alpha,
                                                        const double* __restrict__ V, size_t stride,
                                                        double* __restrict__ out) {
  const int m = idx[blockIdx.y];
  const int n = L.mol_norb[m];
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= n * n) return;
  const size_t o = L.mol_mat_off[m] + t;
  double s = 0.0;
  for (int i = 0; i < r; ++i) s -= alpha[(size_t)m * kMaxRank + i] * V[i * stride + o];
  out[o] = s;
}

inline int elem_blocks(int nmax) { return (nmax * nmax + 255) / 256; }

}  // namespace

extern "C" int pyseqm_ksa_max_rank() { return kMaxRank; }

extern "C" long long pyseqm_fermi_workspace(int nact) {
  return nact < 0 ? -1 : (long long)nact * kFermiIter * (sizeof(double) + 1) + 16;
}

extern "C" int pyseqm_fermi_density(const pyseqm_layout_t* L, const int* idx, int nact, int nmax,
                                    const long long* orb_off, const double* evals, const double* Q, double T,
                                    double kB, double* occ, double* mu, double* D, double* S, void* work,
                                    void* stream) {
  if (!L || nact < 0 || nmax < 2 || nmax > 256 || !(T > 0.0) || !(kB > 0.0) || !work) return PYSEQM_EINVAL;
  if (nact == 0) return PYSEQM_OK;
  hipStream_t s = (hipStream_t)stream;
  const double beta = 1.0 / (kB * T);
  double* mu_hist = static_cast<double*>(work);
  unsigned char* conv = reinterpret_cast<unsigned char*>(mu_hist + (size_t)nact * kFermiIter);
  int* kpick = reinterpret_cast<int*>(conv + (((size_t)nact * kFermiIter + 7) & ~(size_t)7));
  k_fermi_newton<<<nact, 64, 0, s>>>(*L, idx, orb_off, evals, beta, mu_hist, conv);
  k_fermi_pick<<<1, 256, 0, s>>>(nact, conv, kpick);
  k_fermi_occ<<<nact, 256, 0, s>>>(*L, idx, orb_off, evals, beta, kB, mu_hist, kpick, occ, mu, S);
  const int nt = (nmax + 15) / 16;
  k_fermi_density<<<dim3((nt * (nt + 1) / 2 + 3) / 4, nact), 256, 0, s>>>(*L, idx, orb_off, occ, Q, D);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}

extern "C" int pyseqm_block_gemm(const pyseqm_layout_t* L, const int* idx, int nact, int nmax, int ta, int tb,
                                 const double* A, const double* B, double* C, void* stream) {
  if (!L || nact < 0 || nmax < 1) return PYSEQM_EINVAL;
  if (nact == 0) return PYSEQM_OK;
  const int nt = (nmax + 15) / 16;
  const dim3 grid(nt * nt, nact);
  hipStream_t s = (hipStream_t)stream;
  if (ta && tb)
    k_block_gemm<true, true><<<grid, 256, 0, s>>>(*L, idx, A, B, C);
  else if (ta)
    k_block_gemm<true, false><<<grid, 256, 0, s>>>(*L, idx, A, B, C);
  else if (tb)
    k_block_gemm<false, true><<<grid, 256, 0, s>>>(*L, idx, A, B, C);
  else
    k_block_gemm<false, false><<<grid, 256, 0, s>>>(*L, idx, A, B, C);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}

extern "C" int pyseqm_canon_prt(const pyseqm_layout_t* L, const int* idx, int nact, int nmax,
                                const long long* orb_off, const double* evals, const double* mu, double T, double kB,
                                int steps, double* Y, void* stream) {
  if (!L || nact < 0 || nmax < 1 || nmax > 256 || steps < 0 || !(T > 0.0) || !(kB > 0.0)) return PYSEQM_EINVAL;
  if (nact == 0) return PYSEQM_OK;
  hipStream_t s = (hipStream_t)stream;
  const double beta = 1.0 / (kB * T);
  k_canon_elem<<<dim3(elem_blocks(nmax), nact), 256, 0, s>>>(*L, idx, orb_off, evals, mu, beta, steps, Y);
  k_canon_shift<<<nact, 256, 0, s>>>(*L, idx, orb_off, evals, mu, beta, steps, Y);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}

extern "C" int pyseqm_density_response_elem(const pyseqm_layout_t* L, const int* idx, int nact, int nmax,
                                            const long long* orb_off, const double* evals, double* Y, void* stream) {
  if (!L || nact < 0 || nmax < 1) return PYSEQM_EINVAL;
  if (nact == 0) return PYSEQM_OK;
  k_response_elem<<<dim3(elem_blocks(nmax), nact), 256, 0, (hipStream_t)stream>>>(*L, idx, orb_off, evals, Y);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}

extern "C" int pyseqm_block_dot(const pyseqm_layout_t* L, const int* idx, int nact, const double* A,
                                const double* B, double* out, void* stream) {
  if (!L || nact < 0) return PYSEQM_EINVAL;
  if (nact == 0) return PYSEQM_OK;
  k_block_dot<<<nact, 256, 0, (hipStream_t)stream>>>(*L, idx, A, B, out);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}

extern "C" int pyseqm_block_axpy(const pyseqm_layout_t* L, const int* idx, int nact, int nmax, int mode, double s,
                                 const double* c, int cstride, const double* X, double* Y, void* stream) {
  if (!L || nact < 0 || nmax < 1 || mode < 0 || mode > 4 || ((mode == 0 || mode == 1 || mode == 3) && !c))
    return PYSEQM_EINVAL;
  if (nact == 0) return PYSEQM_OK;
  k_block_axpy<<<dim3(elem_blocks(nmax), nact), 256, 0, (hipStream_t)stream>>>(*L, idx, mode, s, c, cstride, X, Y);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}

extern "C" int pyseqm_small_solve(const int* idx, int nact, int r, const double* O, const double* rhs, double* alpha,
                                  void* stream) {
  if (nact < 0 || r < 1 || r > kMaxRank) return PYSEQM_EINVAL;
  if (nact == 0) return PYSEQM_OK;
  k_small_solve<<<(nact + 63) / 64, 64, 0, (hipStream_t)stream>>>(idx, nact, r, O, rhs, alpha);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}

extern "C" int pyseqm_krylov_start(const pyseqm_layout_t* L, const int* idx, int nact, int k, const double* D,
                                   const double* P, double* dDS, double* V, const double* W, long long stride,
                                   void* stream) {
  if (!L || nact < 0 || k < 0 || k >= kMaxRank || stride < 0) return PYSEQM_EINVAL;
  if (nact == 0) return PYSEQM_OK;
  k_krylov_start<<<nact, kKrylovThreads, 0, (hipStream_t)stream>>>(*L, idx, k, D, P, dDS, V, W, (size_t)stride);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}

extern "C" int pyseqm_krylov_fit(const pyseqm_layout_t* L, const int* idx, int nact, int k, const double* V, double* W,
                                 long long stride, const double* dDS, double* O, double* rhs, double* alpha,
                                 void* stream) {
  if (!L || nact < 0 || k < 0 || k >= kMaxRank || stride < 0) return PYSEQM_EINVAL;
  if (nact == 0) return PYSEQM_OK;
  k_krylov_fit<<<nact, kKrylovThreads, 0, (hipStream_t)stream>>>(*L, idx, k, V, W, (size_t)stride, dDS, O, rhs, alpha);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}

extern "C" int pyseqm_krylov_response_ok(int nmax, int steps) {
  return nmax >= 1 && nmax <= 192 && steps >= 0 && steps <= 64 &&
         krylov_lds(nmax, steps) * (long long)sizeof(double) <= 158 * 1024;  // with the static sums, 160 KiB
}

extern "C" int pyseqm_krylov_response(const pyseqm_layout_t* L, const int* idx, int nact, int nmax,
                                      const long long* orb_off, const double* evals, const double* mu, double T,
                                      double kB, int steps, const double* Q, const double* G, int k, const double* V,
                                      double* W, long long stride, const double* dDS, double* O, double* rhs,
                                      double* alpha, void* stream) {
  if (!L || nact < 0 || k < 0 || k >= kMaxRank || stride < 0 || !(T > 0.0) || !(kB > 0.0) ||
      !pyseqm_krylov_response_ok(nmax, steps))
    return PYSEQM_EINVAL;
  if (nact == 0) return PYSEQM_OK;
  const size_t lds = (size_t)krylov_lds(nmax, steps) * sizeof(double);
  k_krylov_response<<<nact, kKrylovThreads, lds, (hipStream_t)stream>>>(*L, idx, orb_off, evals, mu, 1.0 / (kB * T),
                                                                       steps, Q, G, k, V, W, (size_t)stride, dDS, O,
                                                                       rhs, alpha);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}

extern "C" int pyseqm_krylov_combine(const pyseqm_layout_t* L, const int* idx, int nact, int nmax, int r,
                                     const double* alpha, const double* V, long long stride, double* out,
                                     void* stream) {
  if (!L || nact < 0 || nmax < 1 || r < 1 || r > kMaxRank || stride < 0) return PYSEQM_EINVAL;
  if (nact == 0) return PYSEQM_OK;
  k_krylov_combine<<<dim3(elem_blocks(nmax), nact), 256, 0, (hipStream_t)stream>>>(*L, idx, r, alpha, V,
                                                                                   (size_t)stride, out);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}
