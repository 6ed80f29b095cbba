// Pair integrals for MNDO/AM1/PM3 sp atoms on gfx950.
//
// One 64-lane wave per 8x8 pair tile; each lane owns one atom pair and computes, in FP64:
//   * the local-frame two-electron integrals (MOPAC repp point-multipole formulas,
//     two_elec_two_center_int_local_frame.py:18-293),
//   * their rotation to the molecular frame, w = T L T^T with T the 10x10 map from local to
//     molecular orbital-product pairs (same rotation as two_elec_two_center_int.py:1384-1631),
//   * the electron-core attractions e1b/e2a (two_elec_two_center_int.py:1533-1569),
//   * the STO overlap block and the off-diagonal core Hamiltonian H_ij = S_ij (b_i + b_j)/2
//     (diat_overlap_PM6_SP.py:6-444, hcore.py:155-173),
//   * the core-core repulsion (energy.py:91-134).
// Diagonal core-Hamiltonian blocks are summed per atom from per-tile row/column partials in a
// fixed order (deterministic, no atomics).
#include "common.h"

#include <type_traits>

using namespace pyseqm;

namespace {

enum { XX = 0, XH = 1, HH = 2 };  // tile kinds: heavy-heavy, heavy-H, H-H

__device__ constexpr double kTore[19] = {0, 1, 0, 1, 2, 3, 4, 5, 6, 7, 0, 1, 2, 3, 4, 5, 6, 7, 0};
__device__ constexpr int kQn[19] = {0, 1, 1, 2, 2, 2, 2, 2, 2, 2, 2, 3, 3, 3, 3, 3, 3, 3, 3};

// ---------------------------------------------------------------- per-atom setup
// rho1 = 1/(2 ad): hsp = ad/2 - 1/(2 sqrt(4 D1^2 + 1/ad^2)) solved by 5 secant steps from the
// closed-form start (cal_par.py:106-160).
__device__ double secant(int which, double target, double D, double x1) {
  double x2 = x1 + 0.04;
  for (int it = 0; it < 5; ++it) {
    double f1, f2;
    if (which == 1) {
      f1 = 0.5 * x1 - 0.5 / sqrt(4.0 * D * D + 1.0 / (x1 * x1));
      f2 = 0.5 * x2 - 0.5 / sqrt(4.0 * D * D + 1.0 / (x2 * x2));
    } else {
      f1 = 0.25 * x1 - 0.5 / sqrt(4.0 * D * D + 1.0 / (x1 * x1)) + 0.25 / sqrt(8.0 * D * D + 1.0 / (x1 * x1));
      f2 = 0.25 * x2 - 0.5 / sqrt(4.0 * D * D + 1.0 / (x2 * x2)) + 0.25 / sqrt(8.0 * D * D + 1.0 / (x2 * x2));
    }
    const double x3 = fabs(f2 - f1) > 1.0e-16 ? x1 + (x2 - x1) * (target - f1) / (f2 - f1) : x2;
    x1 = x2;
    x2 = x3;
  }
  return x2;
}

// The derived slots (dd, qq, rho0/1/2, tore, qn, Z) of an atom-parameter record from its inputs.
__device__ void derive_atom(double* p, int Z) {
  const double qn = kQn[Z];
  double dd = 0.0, qq = 0.0, r1 = 0.0, r2 = 0.0;
  if (Z > 2) {
    const double zs = p[PAR_ZS], zp = p[PAR_ZP];
    dd = (2.0 * qn + 1.0) * pow(4.0 * zs * zp, qn + 0.5) / pow(zs + zp, 2.0 * qn + 2.0) / sqrt(3.0);
    qq = sqrt((4.0 * qn * qn + 6.0 * qn + 2.0) / 20.0) / zp;
    const double hsp = p[PAR_HSP] / kEV;
    double d1 = cbrt(fabs(hsp) / (dd * dd));
    if (hsp < 0.0) d1 = -d1;
    r1 = 0.5 / secant(1, hsp, dd, d1);
    const double hpp = fmax(0.5 * (p[PAR_GPP] - p[PAR_GP2]), 0.1) / kEV;
    double q1 = pow(fabs(hpp) / 3.0 / (qq * qq * qq * qq), 0.2);
    if (hpp < 0.0) q1 = -q1;
    r2 = 0.5 / secant(2, hpp, qq, q1);
  }
  p[PAR_DD] = dd;
  p[PAR_QQ] = qq;
  p[PAR_RHO0] = 0.5 * kEV / p[PAR_GSS];
  p[PAR_RHO1] = r1;
  p[PAR_RHO2] = r2;
  p[PAR_TORE] = kTore[Z];
  p[PAR_QN] = qn;
  p[PAR_Z] = (double)Z;
}

__global__ void k_atom_setup(pyseqm_layout_t L, double* par) {
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= L.natoms) return;
  derive_atom(par + (size_t)a * PYSEQM_NPAR, L.atom_Z[a]);
}

// ------------------------------------------------------------------ value + derivative
// A function of the pair distance together with its derivative: the force kernels evaluate the
// formulas below once on Duals instead of at displaced geometries.  On plain doubles every helper
// is the operation the integral kernels have always used.
struct Dual {
  double v, d;
};
__device__ inline Dual operator+(Dual a, Dual b) { return {a.v + b.v, a.d + b.d}; }
__device__ inline Dual operator-(Dual a, Dual b) { return {a.v - b.v, a.d - b.d}; }
__device__ inline Dual operator-(Dual a) { return {-a.v, -a.d}; }
__device__ inline Dual operator+(Dual a, double b) { return {a.v + b, a.d}; }
__device__ inline Dual operator+(double a, Dual b) { return {a + b.v, b.d}; }
__device__ inline Dual operator-(Dual a, double b) { return {a.v - b, a.d}; }
__device__ inline Dual operator-(double a, Dual b) { return {a - b.v, -b.d}; }
__device__ inline Dual operator*(double a, Dual b) { return {a * b.v, a * b.d}; }
__device__ inline Dual operator*(Dual a, double b) { return {a.v * b, a.d * b}; }
__device__ inline Dual operator*(Dual a, Dual b) { return {a.v * b.v, fma(a.v, b.d, a.d * b.v)}; }
__device__ inline Dual operator/(Dual a, double b) { return a * (1.0 / b); }
// 1 / x from v_rcp_f64 and two Newton steps, 1 / sqrt(x) from v_rsq_f64 and two (x normal, positive for
// the root): the arguments here are distances and squared distances of atom pairs
__device__ inline double rcp_nr(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
}
__device__ inline double rsq_nr(double x) {
  double r = __builtin_amdgcn_rsq(x);
  r = fma(0.5 * r, fma(-x * r, r, 1.0), r);
  return fma(0.5 * r, fma(-x * r, r, 1.0), r);
}
__device__ inline double inv_root(double x) { return 1.0 / sqrt(x); }
__device__ inline Dual inv_root(Dual x) {
  const double r = rsq_nr(x.v);
  return {r, -0.5 * (r * r * r) * x.d};
}
// a / sqrt(x)
__device__ inline double quot_root(double a, double x) { return a / sqrt(x); }
__device__ inline Dual quot_root(double a, Dual x) { return a * inv_root(x); }
__device__ inline double exp_of(double x) { return exp(x); }
__device__ inline Dual exp_of(Dual x) {
  const double e = exp(x.v);
  return {e, e * x.d};
}
__device__ inline double value_of(double x) { return x; }
__device__ inline double value_of(Dual x) { return x.v; }
__device__ inline double recip(double) { return 0.0; }  // unused: over() divides
__device__ inline Dual recip(Dual x) {
  const double r = rcp_nr(x.v);
  return {r, -(r * r) * x.d};
}
// a / x, given recip(x)
__device__ inline double over(double a, double x, double) { return a / x; }
__device__ inline Dual over(Dual a, Dual, Dual rx) { return a * rx; }
__device__ inline double quot(double a, double x) { return a / x; }
__device__ inline Dual quot(double a, Dual x) { return a * recip(x); }
// x^(k + 1/2), k >= 1, of an exponent product at distance r: on doubles, and where r or x is a Dual
__device__ inline double half_pow(double, double x, int k) { return pow(x, k + 0.5); }
__device__ inline double half_pow(Dual, double x, int k) {
  double p = sqrt(x);
  for (int t = 0; t < k; ++t) p *= x;
  return p;
}
__device__ inline Dual half_pow(double, Dual x, int k) {
  double p = sqrt(x.v);
  for (int t = 1; t < k; ++t) p *= x.v;
  return {p * x.v, (k + 0.5) * p * x.d};
}
__device__ inline double pow_3_2(double x) { return pow(x, 1.5); }
__device__ inline Dual pow_3_2(Dual x) {
  const double q = sqrt(x.v);
  return {x.v * q, 1.5 * q * x.d};
}
// r as a value of its own at each use in a formula on Duals: the A and B integrals of the four exponent
// pairs are then evaluated where they are used, one pair's after another's, and not all together ahead
// of the branches that share them (112 doubles alive, which spilled)
template <class T>
__device__ inline double once(double r) {
  if constexpr (sizeof(T) == sizeof(Dual)) asm volatile("" : "+v"(r));
  return r;
}
template <class T>
__device__ inline Dual once(Dual r) {
  return {once<T>(r.v), r.d};
}
template <class S>
__device__ inline S constant(double x);
template <>
__device__ inline double constant<double>(double x) {
  return x;
}
template <>
__device__ inline Dual constant<Dual>(double x) {
  return {x, 0.0};
}

// ------------------------------------------------------------ local-frame integrals
// 22 heavy-heavy integrals in MOPAC storage order (SS/SS)=0 ... (P*P/P*P)=21, local axis
// sigma pointing from atom j to atom i (two_elec_two_center_int_local_frame.py:126-262).
template <class S>
__device__ inline void local_xx(S r, double da, double db, double qa1, double qb1, double r0a,
                         double r0b, double r1a, double r1b, double r2a, double r2b, S ri[22]) {
  const double e1 = kEV * 0.5, e2 = kEV * 0.25, e3 = kEV * 0.125, e4 = kEV * 0.0625;
  const double qa = 2.0 * qa1, qb = 2.0 * qb1;
  const double aee = (r0a + r0b) * (r0a + r0b), ade = (r1a + r0b) * (r1a + r0b);
  const double aqe = (r2a + r0b) * (r2a + r0b), aed = (r0a + r1b) * (r0a + r1b);
  const double aeq = (r0a + r2b) * (r0a + r2b), axx = (r1a + r1b) * (r1a + r1b);
  const double adq = (r1a + r2b) * (r1a + r2b), aqd = (r2a + r1b) * (r2a + r1b);
  const double aqq = (r2a + r2b) * (r2a + r2b);
  const S r2 = r * r;
  auto inv = [](S x) { return inv_root(x); };
  const S ee = kEV * inv(r2 + aee);
  const S dze = -e1 * inv((r + da) * (r + da) + ade) + e1 * inv((r - da) * (r - da) + ade);
  const S c6 = e1 * inv(r2 + aqe);
  const S qzze = e2 * inv((r - qa) * (r - qa) + aqe) + e2 * inv((r + qa) * (r + qa) + aqe) - c6;
  const S qxxe = e1 * inv(r2 + qa * qa + aqe) - c6;
  const S edz = -e1 * inv((r - db) * (r - db) + aed) + e1 * inv((r + db) * (r + db) + aed);
  const S c12 = e1 * inv(r2 + aeq);
  const S eqzz = e2 * inv((r - qb) * (r - qb) + aeq) + e2 * inv((r + qb) * (r + qb) + aeq) - c12;
  const S eqxx = e1 * inv(r2 + qb * qb + aeq) - c12;
  const S t20 = e2 * inv((r + da) * (r + da) + adq), t22 = e2 * inv((r - da) * (r - da) + adq);
  const S t24 = e2 * inv((r - db) * (r - db) + aqd), t26 = e2 * inv((r + db) * (r + db) + aqd);
  const S t36 = e2 * inv(r2 + aqq), t39 = e2 * inv(r2 + qa * qa + aqq), t40 = e2 * inv(r2 + qb * qb + aqq);
  const S t42 = e3 * inv((r - qb) * (r - qb) + aqq), t44 = e3 * inv((r + qb) * (r + qb) + aqq);
  const S t46 = e3 * inv((r + qa) * (r + qa) + aqq), t48 = e3 * inv((r - qa) * (r - qa) + aqq);
  auto sq = [](auto x) { return x * x; };
  ri[0] = ee;
  ri[1] = -dze;
  ri[2] = ee + qzze;
  ri[3] = ee + qxxe;
  ri[4] = -edz;
  ri[5] = e2 * inv(sq(r + da - db) + axx) + e2 * inv(sq(r - da + db) + axx) -
          e2 * inv(sq(r - da - db) + axx) - e2 * inv(sq(r + da + db) + axx);
  ri[6] = e1 * inv(r2 + sq(da - db) + axx) - e1 * inv(r2 + sq(da + db) + axx);
  ri[7] = -edz + e3 * inv(sq(r + qa - db) + aqd) - e3 * inv(sq(r + qa + db) + aqd) +
          e3 * inv(sq(r - qa - db) + aqd) - e3 * inv(sq(r - qa + db) + aqd) - t24 + t26;
  ri[8] = -edz - t24 + e2 * inv(sq(r - db) + qa * qa + aqd) + t26 - e2 * inv(sq(r + db) + qa * qa + aqd);
  ri[9] = e2 * inv(sq(qa1 - db) + sq(r + qa1) + aqd) - e2 * inv(sq(qa1 - db) + sq(r - qa1) + aqd) -
          e2 * inv(sq(qa1 + db) + sq(r + qa1) + aqd) + e2 * inv(sq(qa1 + db) + sq(r - qa1) + aqd);
  ri[10] = ee + eqzz;
  ri[11] = ee + eqxx;
  ri[12] = -dze + e3 * inv(sq(r + da - qb) + adq) - e3 * inv(sq(r - da - qb) + adq) +
           e3 * inv(sq(r + da + qb) + adq) - e3 * inv(sq(r - da + qb) + adq) + t22 - t20;
  ri[13] = -dze - t20 + e2 * inv(sq(r + da) + qb * qb + adq) + t22 - e2 * inv(sq(r - da) + qb * qb + adq);
  ri[14] = e2 * inv(sq(da - qb1) + sq(r - qb1) + adq) - e2 * inv(sq(da - qb1) + sq(r + qb1) + adq) -
           e2 * inv(sq(da + qb1) + sq(r - qb1) + adq) + e2 * inv(sq(da + qb1) + sq(r + qb1) + adq);
  ri[15] = ee + eqzz + qzze + e4 * inv(sq(r + qa - qb) + aqq) + e4 * inv(sq(r + qa + qb) + aqq) +
           e4 * inv(sq(r - qa - qb) + aqq) + e4 * inv(sq(r - qa + qb) + aqq) - t48 - t46 - t42 - t44 + t36;
  ri[16] = ee + eqzz + qxxe + e3 * inv(sq(r - qb) + qa * qa + aqq) + e3 * inv(sq(r + qb) + qa * qa + aqq) -
           t42 - t44 - t39 + t36;
  ri[17] = ee + eqxx + qzze + e3 * inv(sq(r + qa) + qb * qb + aqq) + e3 * inv(sq(r - qa) + qb * qb + aqq) -
           t46 - t48 - t40 + t36;
  const S qxxqxx = e3 * inv(r2 + sq(qa - qb) + aqq) + e3 * inv(r2 + sq(qa + qb) + aqq) - t39 - t40 + t36;
  ri[18] = ee + eqxx + qxxe + qxxqxx;
  const double dm = sq(qa1 - qb1), dp = sq(qa1 + qb1);
  ri[19] = e3 * inv(sq(r + qa1 - qb1) + dm + aqq) - e3 * inv(sq(r + qa1 + qb1) + dm + aqq) -
           e3 * inv(sq(r - qa1 - qb1) + dm + aqq) + e3 * inv(sq(r - qa1 + qb1) + dm + aqq) -
           e3 * inv(sq(r + qa1 - qb1) + dp + aqq) + e3 * inv(sq(r + qa1 + qb1) + dp + aqq) +
           e3 * inv(sq(r - qa1 - qb1) + dp + aqq) - e3 * inv(sq(r - qa1 + qb1) + dp + aqq);
  const S qxxqyy = e2 * inv(r2 + qa * qa + qb * qb + aqq) - t39 - t40 + t36;
  ri[20] = ee + eqxx + qxxe + qxxqyy;
  ri[21] = 0.5 * (qxxqxx - qxxqyy);
}

// 4 heavy-H integrals (two_elec_two_center_int_local_frame.py:90-107)
template <class S>
__device__ inline void local_xh(S r, double da, double qa1, double r0a, double r1a, double r2a,
                         double r0b, S ri[4]) {
  const double e1 = kEV * 0.5, e2 = kEV * 0.25;
  const double qa = 2.0 * qa1;
  const double aee = (r0a + r0b) * (r0a + r0b), ade = (r1a + r0b) * (r1a + r0b);
  const double aqe = (r2a + r0b) * (r2a + r0b);
  const S ee = quot_root(kEV, r * r + aee);
  const S c = quot_root(e1, r * r + aqe);
  ri[0] = ee;
  ri[1] = quot_root(e1, (r + da) * (r + da) + ade) - quot_root(e1, (r - da) * (r - da) + ade);
  ri[2] = ee + quot_root(e2, (r + qa) * (r + qa) + aqe) + quot_root(e2, (r - qa) * (r - qa) + aqe) - c;
  ri[3] = ee + quot_root(e1, r * r + qa * qa + aqe) - c;
}

// Rotation with R v = e_x built from the quaternion of v (two_elec_two_center_int.py:1576-1631),
// including its antipodal fallback (|1 + v_x| < 1e-7 -> constant 180 deg turn about z).
// mode 0: as the reference; 1: never take the fallback (smooth in v); 2: always the fallback.
// Gradients take 1 or 2 by quat_flips, which reproduces the reference's autograd derivative (zero
// frame derivative inside the fallback cone).
__device__ inline bool quat_flips(double vx) { return fabs(1.0 + vx) < 1.0e-7; }

__device__ inline void quat_frame(double vx, double vy, double vz, double R[3][3], int mode = 0) {
  double qy = vz, qz = -vy, qw = 1.0 + vx;
  if (mode == 2 || (mode == 0 && fabs(qw) < 1.0e-7)) {
    qy = 0.0;
    qz = 1.0;
    qw = 0.0;
  }
  const double n = 1.0 / sqrt(qy * qy + qz * qz + qw * qw);
  qy *= n;
  qz *= n;
  qw *= n;
  R[0][0] = 1.0 - 2.0 * (qy * qy + qz * qz);
  R[0][1] = -2.0 * (qz * qw);
  R[0][2] = 2.0 * (qy * qw);
  R[1][0] = 2.0 * (qz * qw);
  R[1][1] = 1.0 - 2.0 * (qz * qz);
  R[1][2] = 2.0 * (qy * qz);
  R[2][0] = -2.0 * (qy * qw);
  R[2][1] = 2.0 * (qy * qz);
  R[2][2] = 1.0 - 2.0 * (qy * qy);
}

// T[k][p]: coefficient of local pair p = (a>=b) in molecular pair k = (mu>=nu), where
// molecular p_m = sum_a R[a][m] * local_(1+a).
__device__ inline void pair_map(const double R[3][3], double T[10][10]) {
  double U[4][4];
  U[0][0] = 1.0;
#pragma unroll
  for (int a = 1; a < 4; ++a) U[0][a] = U[a][0] = 0.0;
#pragma unroll
  for (int m = 0; m < 3; ++m)
#pragma unroll
    for (int a = 0; a < 3; ++a) U[1 + m][1 + a] = R[a][m];
#pragma unroll
  for (int k = 0; k < 10; ++k)
#pragma unroll
    for (int p = 0; p < 10; ++p) {
      const int mu = kTriI[k], nu = kTriJ[k], a = kTriI[p], b = kTriJ[p];
      T[k][p] = U[mu][a] * U[nu][b] + (a != b ? U[mu][b] * U[nu][a] : 0.0);
    }
}

// Local tensor over local orbital-product pairs (s,s)=0 (sig,s)=1 (sig,sig)=2 (pi,s)=3
// (pi,sig)=4 (pi,pi)=5 (pi',s)=6 (pi',sig)=7 (pi',pi)=8 (pi',pi')=9.
__device__ inline void local_tensor(const double ri[22], double Lm[10][10]) {
#pragma unroll
  for (int p = 0; p < 10; ++p)
#pragma unroll
    for (int q = 0; q < 10; ++q) Lm[p][q] = 0.0;
  Lm[0][0] = ri[0];  Lm[0][1] = ri[4];  Lm[0][2] = ri[10]; Lm[0][5] = ri[11]; Lm[0][9] = ri[11];
  Lm[1][0] = ri[1];  Lm[1][1] = ri[5];  Lm[1][2] = ri[12]; Lm[1][5] = ri[13]; Lm[1][9] = ri[13];
  Lm[2][0] = ri[2];  Lm[2][1] = ri[7];  Lm[2][2] = ri[15]; Lm[2][5] = ri[17]; Lm[2][9] = ri[17];
  Lm[3][3] = ri[6];  Lm[3][4] = ri[14];
  Lm[4][3] = ri[9];  Lm[4][4] = ri[19];
  Lm[5][0] = ri[3];  Lm[5][1] = ri[8];  Lm[5][2] = ri[16]; Lm[5][5] = ri[18]; Lm[5][9] = ri[20];
  Lm[6][6] = ri[6];  Lm[6][7] = ri[14];
  Lm[7][6] = ri[9];  Lm[7][7] = ri[19];
  Lm[8][8] = ri[21];
  Lm[9][0] = ri[3];  Lm[9][1] = ri[8];  Lm[9][2] = ri[16]; Lm[9][5] = ri[20]; Lm[9][9] = ri[18];
}

// ------------------------------------------------------------------- STO overlaps
// A_k(x) = int_1^inf t^k e^{-xt} dt and B_k(x) = int_-1^1 t^k e^{-xt} dt, k = 0..6, with the
// reference's recurrences / truncated series (diat_overlap_PM6_SP.py:464-670).
template <class S>
__device__ inline void aint7(S x, S a[7]) {
  if (value_of(x) == 0.0) {
#pragma unroll
    for (int k = 0; k < 7; ++k) a[k] = constant<S>(0.0);
    return;
  }
  const S rx = recip(x);
  a[0] = over(exp_of(-x), x, rx);
#pragma unroll
  for (int k = 1; k < 7; ++k) a[k] = a[0] + over((double)k * a[k - 1], x, rx);
}

// Branch of bint7 at argument x: 2 recurrence (|x| > 0.5), 1 truncated series, 0 x ~ 0.
__device__ inline int bint_branch(double x) {
  const double ax = fabs(x);
  return ax > 0.5 ? 2 : (ax > 1.0e-6 ? 1 : 0);
}

template <class S>
__device__ inline void bint7(S x, S b[7]) {
  const int br = bint_branch(value_of(x));
  if (br == 2) {
    const S rx = recip(x);
    const S tx = over(exp_of(x), x, rx), tmx = over(-exp_of(-x), x, rx);
    b[0] = tx + tmx;
#pragma unroll
    for (int k = 1; k < 7; ++k) b[k] = ((k & 1) ? -tx : tx) + tmx + over((double)k * b[k - 1], x, rx);
  } else if (br == 1) {
    const S x2 = x * x, x3 = x2 * x, x4 = x2 * x2, x5 = x4 * x, x6 = x4 * x2;
    b[0] = 2.0 + x2 / 3.0 + x4 / 60.0 + x6 / 2520.0;
    b[2] = 2.0 / 3.0 + x2 / 5.0 + x4 / 84.0 + x6 / 3240.0;
    b[4] = 2.0 / 5.0 + x2 / 7.0 + x4 / 108.0 + x6 / 3960.0;
    b[6] = 2.0 / 7.0 + x2 / 9.0 + x4 / 132.0 + x6 / 4680.0;
    b[1] = -2.0 / 3.0 * x - x3 / 15.0 - x5 / 420.0;
    b[3] = -2.0 / 5.0 * x - x3 / 21.0 - x5 / 540.0;
    b[5] = -2.0 / 7.0 * x - x3 / 27.0 - x5 / 660.0;
  } else {
    const double at0[7] = {2.0, 0.0, 2.0 / 3.0, 0.0, 2.0 / 5.0, 0.0, 2.0 / 7.0};
#pragma unroll
    for (int k = 0; k < 7; ++k) b[k] = constant<S>(at0[k]);
  }
}

__device__ inline int jcall_of(int qi, int qj) {
  if (qi == 1 && qj == 1) return 2;
  if (qi == 2 && qj == 1) return 3;
  if (qi == 2 && qj == 2) return 4;
  if (qi == 3 && qj == 1) return 431;
  if (qi == 3 && qj == 2) return 5;
  if (qi == 3 && qj == 3) return 6;
  return 0;
}

// S[0..4] = S111 (s|s), S211 (p_sig(i)|s(j)), S121, S221, S222 in the diatomic frame
// (diat_overlap_PM6_SP.py:84-345).  za/zb = (zeta_s, zeta_p) of atoms i / j.
// T is the type of the results: Dual where r or the exponents are.  KIND (XX, XH, HH) limits the code
// to the formulas that a tile of that kind can meet.
template <class T, int KIND, class Rt, class Zt>
__device__ inline void overlap_local(int jc, Rt r, Zt zas, Zt zap, Zt zbs, Zt zbp, bool need_p_i, T S[5]) {
  S[0] = S[1] = S[2] = S[3] = S[4] = constant<T>(0.0);
  T A[7], B[7];
  const double s3 = 1.7320508075688772;
  const double s10 = 3.1622776601683795, s30 = 5.477225575051661;
  auto AB = [&](Zt z1, Zt z2) {
    const Rt h = 0.5 * once<T>(r);
    aint7<T>(h * (z1 + z2), A);
    bint7<T>(h * (z1 - z2), B);
  };
  if (KIND == HH && jc == 2) {
    AB(zas, zbs);
    S[0] = pow_3_2(zas * zbs * r * r) * (A[2] * B[0] - B[2] * A[0]) / 4.0;
  } else if (KIND == XH && jc == 3) {
    const Rt r4 = r * r * r * r;
    AB(zas, zbs);
    S[0] = half_pow(r, zbs, 1) * half_pow(r, zas, 2) * r4 * (A[3] * B[0] - B[3] * A[0] + A[2] * B[1] - B[2] * A[1]) / (s3 * 8.0);
    if (need_p_i) {
      AB(zap, zbs);
      S[1] = half_pow(r, zbs, 1) * half_pow(r, zap, 2) * r4 * (A[2] * B[0] - B[2] * A[0] + A[3] * B[1] - B[3] * A[1]) / 8.0;
    }
  } else if (KIND == XX && jc == 4) {
    const Rt r5 = r * r * r * r * r;
    AB(zas, zbs);
    S[0] = half_pow(r, zbs * zas, 2) * r5 * (A[4] * B[0] + B[4] * A[0] - 2.0 * A[2] * B[2]) / 48.0;
    AB(zap, zbs);
    S[1] = half_pow(r, zbs * zap, 2) * r5 *
           (A[3] * (B[0] - B[2]) - A[1] * (B[2] - B[4]) + B[3] * (A[0] - A[2]) - B[1] * (A[2] - A[4])) /
           (16.0 * s3);
    AB(zas, zbp);
    S[2] = half_pow(r, zbp * zas, 2) * r5 *
           (A[3] * (B[0] - B[2]) - A[1] * (B[2] - B[4]) - B[3] * (A[0] - A[2]) + B[1] * (A[2] - A[4])) /
           (16.0 * s3);
    AB(zap, zbp);
    const T w = half_pow(r, zbp * zap, 2) * r5 / 16.0;
    S[3] = -w * (B[2] * (A[4] + A[0]) - A[2] * (B[4] + B[0]));
    S[4] = 0.5 * w * (A[4] * (B[0] - B[2]) - B[4] * (A[0] - A[2]) - A[2] * B[0] + B[2] * A[0]);
  } else if (KIND == XH && jc == 431) {
    const Rt r5 = r * r * r * r * r;
    AB(zas, zbs);
    S[0] = half_pow(r, zbs, 1) * half_pow(r, zas, 3) * r5 *
           (A[4] * B[0] + 2.0 * B[1] * A[3] - 2.0 * A[1] * B[3] - B[4] * A[0]) / (s10 * 24.0);
    if (need_p_i) {
      AB(zap, zbs);
      S[1] = half_pow(r, zbs, 1) * half_pow(r, zap, 3) * r5 *
             (A[3] * (B[0] + B[2]) - A[1] * (B[4] + B[2]) + B[1] * (A[2] + A[4]) - B[3] * (A[2] + A[0])) /
             (8.0 * s30);
    }
  } else if (KIND == XX && jc == 5) {
    const Rt r6 = r * r * r * r * r * r;
    AB(zas, zbs);
    S[0] = half_pow(r, zbs, 2) * half_pow(r, zas, 3) * r6 *
           (A[5] * B[0] + B[1] * A[4] - 2.0 * B[2] * A[3] - 2.0 * A[2] * B[3] + B[4] * A[1] + B[5] * A[0]) /
           (s30 * 48.0);
    AB(zap, zbs);
    S[1] = half_pow(r, zbs, 2) * half_pow(r, zap, 3) * r6 *
           (A[4] * B[0] + B[1] * A[5] - 2.0 * B[3] * A[3] - 2.0 * A[2] * B[2] + A[1] * B[5] + A[0] * B[4]) /
           (48.0 * s10);
    AB(zas, zbp);
    S[2] = half_pow(r, zbp, 2) * half_pow(r, zas, 3) * r6 *
           ((A[4] * B[0] - A[5] * B[1]) + 2.0 * (A[3] * B[1] - A[4] * B[2]) - 2.0 * (A[1] * B[3] - A[2] * B[4]) -
            (A[0] * B[4] - A[1] * B[5])) /
           (48.0 * s10);
    AB(zap, zbp);
    const T pre = half_pow(r, zbp, 2) * half_pow(r, zap, 3) * r6;
    S[3] = pre *
           ((A[3] * B[0] - A[5] * B[2]) + (A[2] * B[1] - A[4] * B[3]) - (A[1] * B[2] - A[3] * B[4]) -
            (A[0] * B[3] - A[2] * B[5])) /
           (16.0 * s30);
    S[4] = pre *
           ((A[5] - A[3]) * (B[0] - B[2]) + (A[4] - A[2]) * (B[1] - B[3]) - (A[3] - A[1]) * (B[2] - B[4]) -
            (A[2] - A[0]) * (B[3] - B[5])) /
           (32.0 * s30);
  } else if (KIND == XX && jc == 6) {
    const Rt r7 = r * r * r * r * r * r * r;
    AB(zas, zbs);
    S[0] = half_pow(r, zbs * zas, 3) * r7 * (A[6] * B[0] - 3.0 * B[2] * A[4] + 3.0 * A[2] * B[4] - A[0] * B[6]) / 1440.0;
    AB(zap, zbs);
    S[1] = half_pow(r, zbs * zap, 3) * r7 *
           ((A[5] * B[0] + A[6] * B[1]) + (-A[4] * B[1] - A[5] * B[2]) - 2.0 * (A[3] * B[2] + A[4] * B[3]) -
            2.0 * (-A[2] * B[3] - A[3] * B[4]) + (A[1] * B[4] + A[2] * B[5]) + (-A[0] * B[5] - A[1] * B[6])) /
           (480.0 * s3);
    AB(zas, zbp);
    S[2] = half_pow(r, zbp * zas, 3) * r7 *
           ((A[5] * B[0] - A[6] * B[1]) + (A[4] * B[1] - A[5] * B[2]) - 2.0 * (A[3] * B[2] - A[4] * B[3]) -
            2.0 * (A[2] * B[3] - A[3] * B[4]) + (A[1] * B[4] - A[2] * B[5]) + (A[0] * B[5] - A[1] * B[6])) /
           (480.0 * s3);
    AB(zap, zbp);
    const T pre = half_pow(r, zbp, 3) * half_pow(r, zap, 3) * r7;
    S[3] = pre * ((A[4] * B[0] - A[6] * B[2]) - 2.0 * (A[2] * B[2] - A[4] * B[4]) + (A[0] * B[4] - A[2] * B[6])) / 480.0;
    S[4] = pre *
           ((A[6] - A[4]) * (B[0] - B[2]) - 2.0 * (A[4] - A[2]) * (B[2] - B[4]) + (A[2] - A[0]) * (B[4] - B[6])) /
           960.0;
  }
}

// --------------------------------------------------------------- core-core repulsion
template <class S>
__device__ inline S core_repulsion(int method, int Zi, int Zj, S rbohr, S gam, const double* pi,
                           const double* pj) {
  const S ra = rbohr * kA0;
  const double ti = pi[PAR_TORE], tj = pj[PAR_TORE];
  const S t1 = ti * tj * gam;
  S t2 = exp_of(-pi[PAR_ALPHA] * ra);
  if ((Zi == 7 || Zi == 8) && Zj == 1) t2 = t2 * ra;
  const S t3 = exp_of(-pj[PAR_ALPHA] * ra);
  S e = t1 * (1.0 + t2 + t3);
  const int ng = method == PYSEQM_AM1 ? 4 : (method == PYSEQM_PM3 ? 2 : 0);
  if (ng) {
    S g = constant<S>(0.0);
    for (int k = 0; k < ng; ++k) {
      const double* ki = pi + PAR_GAUSS + 3 * k;
      const double* kj = pj + PAR_GAUSS + 3 * k;
      g = g + ki[0] * exp_of(-ki[1] * (ra - ki[2]) * (ra - ki[2]));
      g = g + kj[0] * exp_of(-kj[1] * (ra - kj[2]) * (ra - kj[2]));
    }
    e = e + quot(ti * tj, ra) * g;
  }
  return e;
}

struct PairGeom {
  double x[3];  // unit vector i -> j
  double r;     // bohr
};

__device__ inline PairGeom geom_from_vector(double dx, double dy, double dz) {
  PairGeom g;
  const double d = sqrt(dx * dx + dy * dy + dz * dz);
  g.x[0] = dx / d;
  g.x[1] = dy / d;
  g.x[2] = dz / d;
  g.r = d * (1.0 / kA0);
  return g;
}

__device__ inline PairGeom pair_geom(const double* coords, int i, int j) {
  return geom_from_vector(coords[3 * j] - coords[3 * i], coords[3 * j + 1] - coords[3 * i + 1],
                          coords[3 * j + 2] - coords[3 * i + 2]);
}

// Molecular-frame two-electron integrals of a heavy-heavy pair, column by column:
// fn(k, l, (mu nu|la si)) for k = tril(mu, nu) on atom i and l = tril(la, si) on atom j.
template <class Fn>
__device__ inline void xx_integrals(const PairGeom& g, const double* pi, const double* pj, Fn&& fn) {
  double ri[22];
  local_xx(g.r, pi[PAR_DD], pj[PAR_DD], pi[PAR_QQ], pj[PAR_QQ], pi[PAR_RHO0], pj[PAR_RHO0], pi[PAR_RHO1],
           pj[PAR_RHO1], pi[PAR_RHO2], pj[PAR_RHO2], ri);
  double R[3][3];
  quat_frame(-g.x[0], -g.x[1], -g.x[2], R);
  double T[10][10], Lm[10][10];
  pair_map(R, T);
  local_tensor(ri, Lm);
#pragma unroll
  for (int l = 0; l < 10; ++l) {
    double v[10];
#pragma unroll
    for (int p = 0; p < 10; ++p) {
      double s = 0.0;
#pragma unroll
      for (int q = 0; q < 10; ++q) s += Lm[p][q] * T[l][q];
      v[p] = s;
    }
#pragma unroll
    for (int k = 0; k < 10; ++k) {
      double s = 0.0;
#pragma unroll
      for (int p = 0; p < 10; ++p) s += T[k][p] * v[p];
      fn(k, l, s);
    }
  }
}

// Heavy-H integrals (mu nu|s s), k = tril(mu, nu) on the heavy atom i.
template <class Fn>
__device__ inline void xh_integrals(const PairGeom& g, const double* pi, const double* pj, Fn&& fn) {
  double ri[4];
  local_xh(g.r, pi[PAR_DD], pi[PAR_QQ], pi[PAR_RHO0], pi[PAR_RHO1], pi[PAR_RHO2], pj[PAR_RHO0], ri);
  double R[3][3];
  quat_frame(-g.x[0], -g.x[1], -g.x[2], R);
  double T[10][10];
  pair_map(R, T);
#pragma unroll
  for (int k = 0; k < 10; ++k) fn(k, T[k][0] * ri[0] + T[k][1] * ri[1] + T[k][2] * ri[2] + (T[k][5] + T[k][9]) * ri[3]);
}

__device__ inline double hh_integral(const PairGeom& g, const double* pi, const double* pj) {
  return kEV / sqrt(g.r * g.r + (pi[PAR_RHO0] + pj[PAR_RHO0]) * (pi[PAR_RHO0] + pj[PAR_RHO0]));
}

// Off-diagonal core block H_ij[a][b] = S_ij[a][b] (beta_a(i) + beta_b(j)) / 2 for NI x NJ orbitals.
template <int NI, int NJ>
__device__ inline void core_block(const PairGeom& g, const double* pi, const double* pj, double Hb[4][4]) {
  double di[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) di[a][b] = 0.0;
  if (g.r <= kOverlapCut) {
    const int jc = jcall_of((int)pi[PAR_QN], (int)pj[PAR_QN]);  // validated on the host
    double S[5];
    overlap_local<double, NJ == 4 ? XX : NI == 4 ? XH : HH>(jc, g.r, pi[PAR_ZS], pi[PAR_ZP], pj[PAR_ZS], pj[PAR_ZP],
                                                             NI == 4, S);
    double Rp[3][3];
    quat_frame(g.x[0], g.x[1], g.x[2], Rp);
    di[0][0] = S[0];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      di[1 + m][0] = S[1] * Rp[0][m];
      di[0][1 + m] = -S[2] * Rp[0][m];
    }
    if (NJ == 4) {
      const double D[3] = {-S[3], S[4], S[4]};
#pragma unroll
      for (int m = 0; m < 3; ++m)
#pragma unroll
        for (int n = 0; n < 3; ++n)
          di[1 + m][1 + n] = Rp[0][m] * D[0] * Rp[0][n] + Rp[1][m] * D[1] * Rp[1][n] + Rp[2][m] * D[2] * Rp[2][n];
    }
  }
  const double bi[4] = {pi[PAR_BS], pi[PAR_BP], pi[PAR_BP], pi[PAR_BP]};
  const double bj[4] = {pj[PAR_BS], pj[PAR_BP], pj[PAR_BP], pj[PAR_BP]};
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) Hb[a][b] = (a < NI && b < NJ) ? di[a][b] * 0.5 * (bi[a] + bj[b]) : 0.0;
}

// ------------------------------------------------------------------- tile kernels

// The kernels over pair tiles come per kind of tile (first tile tile_base, its integrals or nothing in w) and as
// ALL: one launch over the three kinds in that order.  A launch per kind lets light tiles run at their own
// register count (up to 8 waves per SIMD, heavy-heavy ones 1); where all tiles fit the chip about at once
// the launches only wait for each other.  Integrals and forces (us, per kind -> ALL) of n alkanes of 2-30 carbons:
// n = 1 38.6 -> 25.0 and 28.7 -> 17.0; 64 (2116 tiles) 52.5 -> 31.1 and 36.5 -> 21.3; 128 (4270) 55.1 -> 47.5 and
// 39.7 -> 35.0; 256 (8548) 91.7 -> 83.5 and 66.7 -> 63.6; 512 (17110) 137 -> 149 and 102 -> 119: ALL up to 8192,
// with at most 6144 light ones (800 / 2400 / 4800 tiles heavy-heavy / heavy-H / H-H 63.4 -> 65.7 and 48.3 -> 52.7;
// 2700 each 132 -> 120 and 88 -> 84).  Without heavy-heavy tiles, whose latency the light ones fill, they lose
// sooner: 500 + 500 25.2 -> 18.8 and 21.0 -> 15.8, 1500 + 1500 30.9 -> 30.3 and 24.3 -> 24.3, 4000 + 4000 39.7 ->
// 59.9 and 33.7 -> 50.4; 8000 H-H alone 22.3 -> 40.1 and 21.4 -> 38.0.
constexpr int ALL = 3;
constexpr int kMergeTiles = 8192, kMergeLight = 6144, kMergeNoHeavy = 3072;
inline bool merge_kinds(const pyseqm_layout_t* L) {
  const long long n0 = L->ntile[0], light = (long long)L->ntile[1] + L->ntile[2];
  return n0 > 0 ? n0 + light <= kMergeTiles && light <= kMergeLight : L->ntile[1] > 0 && light <= kMergeNoHeavy;
}
// f(kind as a constant, tile) for this block's tile
template <int KIND, class Fn>
__device__ __forceinline__ void for_tile(const pyseqm_layout_t& L, int tile_base, Fn f) {
  if constexpr (KIND != ALL) {
    f(std::integral_constant<int, KIND>(), tile_base + xcd_run(blockIdx.x, gridDim.x));
  } else {
    const int n0 = L.ntile[0], n1 = L.ntile[1], n2 = L.ntile[2], b = blockIdx.x;
    if (b < n0)
      f(std::integral_constant<int, XX>(), xcd_run(b, n0));
    else if (b < n0 + n1)
      f(std::integral_constant<int, XH>(), n0 + xcd_run(b - n0, n1));
    else
      f(std::integral_constant<int, HH>(), n0 + n1 + xcd_run(b - n0 - n1, n2));
  }
}

template <int KIND>
__device__ __forceinline__ void pair_tile(const pyseqm_layout_t& L, int method, int tile,
                                          const double* __restrict__ coords, const double* __restrict__ par,
                                          double* __restrict__ wout, double* __restrict__ H,
                                          double* __restrict__ part, double* __restrict__ enuc_tile,
                                          double* __restrict__ enuc_pair, const int* __restrict__ pair_ref) {
  const int lane = threadIdx.x;
  const Tile t = load_tile(L.tiles, tile);
  int i, j;
  const bool valid = lane_pair(t, lane, i, j);
  constexpr int NR = KIND == HH ? 1 : 10;
  constexpr int NC = KIND == XX ? 10 : 1;
  constexpr int NI = KIND == HH ? 1 : 4;
  constexpr int NJ = KIND == XX ? 4 : 1;
  double rowv[NR], colv[NC];
#pragma unroll
  for (int k = 0; k < NR; ++k) rowv[k] = 0.0;
#pragma unroll
  for (int k = 0; k < NC; ++k) colv[k] = 0.0;
  double en = 0.0;
  constexpr int NW = KIND == XX ? 100 : (KIND == XH ? 10 : 1);
  const int S = tile_wstride(t);
  double* wt = wout + L.tile_woff[tile] + (valid ? lane_rank(t, lane) : 0);

  if (valid) {
    const double* pi = par + (size_t)i * PYSEQM_NPAR;
    const double* pj = par + (size_t)j * PYSEQM_NPAR;
    const PairGeom g = pair_geom(coords, i, j);
    const double ti = pi[PAR_TORE], tj = pj[PAR_TORE];
    double gam = 0.0;
    if constexpr (KIND == XX) {
      xx_integrals(g, pi, pj, [&](int k, int l, double w) {
        wt[(size_t)(k * 10 + l) * S] = w;
        if (l == 0) rowv[k] = -tj * w;  // e1b: electrons of i, core of j
        if (k == 0) colv[l] = -ti * w;  // e2a: electrons of j, core of i
        if (k == 0 && l == 0) gam = w;
      });
    } else if constexpr (KIND == XH) {
      xh_integrals(g, pi, pj, [&](int k, double w) {
        wt[(size_t)k * S] = w;
        rowv[k] = -tj * w;
        if (k == 0) gam = w;
      });
      colv[0] = -ti * gam;
    } else {
      gam = hh_integral(g, pi, pj);
      wt[0] = gam;
      rowv[0] = -tj * gam;
      colv[0] = -ti * gam;
    }
    double Hb[4][4];
    core_block<NI, NJ>(g, pi, pj, Hb);
    const long long mo = L.mol_mat_off[t.mol];
    const int norb = L.mol_norb[t.mol];
    const int ai = L.atom_ao[i], aj = L.atom_ao[j];
    double* Hm = H + mo;
#pragma unroll
    for (int a = 0; a < NI; ++a)
#pragma unroll
      for (int b = 0; b < NJ; ++b) {
        Hm[(size_t)(ai + a) * norb + aj + b] = Hb[a][b];
        Hm[(size_t)(aj + b) * norb + ai + a] = Hb[a][b];
      }
    en = core_repulsion(method, (int)pi[PAR_Z], (int)pj[PAR_Z], g.r, gam, pi, pj);
    if (enuc_pair) enuc_pair[pair_ref[(size_t)tile * 64 + lane]] = en;
  }
  write_partials_c(part, L, tile, lane, rowv, colv);
  const double es = wave64(en);  // every lane active here
  if (lane == 0) enuc_tile[tile] = es;
}

template <int KIND>
__global__ __launch_bounds__(64) void k_pair_tiles(pyseqm_layout_t L, int method, int tile_base,
                                                   const double* __restrict__ coords,
                                                   const double* __restrict__ par, double* __restrict__ w_xx,
                                                   double* __restrict__ w_xh, double* __restrict__ w_hh,
                                                   double* __restrict__ H, double* __restrict__ part,
                                                   double* __restrict__ enuc_tile, double* __restrict__ enuc_pair,
                                                   const int* __restrict__ pair_ref) {
  for_tile<KIND>(L, tile_base, [&](auto kind, int tile) {
    constexpr int K = decltype(kind)::value;
    pair_tile<K>(L, method, tile, coords, par, K == XX ? w_xx : (K == XH ? w_xh : w_hh), H, part, enuc_tile, enuc_pair,
                 pair_ref);
  });
}

// Hellmann-Feynman pair energy at fixed density: the part of 0.5 sum P (H + F) + E_nuc that
// depends on the geometry of pair (i, j) (basics.py:1315-1336 differentiates the same energy with
// scf_backward = 0): 2 sum P_ij H_ij + sum P_ii e1b + sum P_jj e2a + sum P_ii P_jj (..|..)
// - 1/2 sum P_ij P_ij (..|..) + E_nuc(i, j).
// With XL = true the energy is the extended-Lagrangian one, sum D F(P) - 1/2 (F(P) - H) P + E_nuc
// (energy.py:76-88, differentiated at fixed D and P by xlbomd.py:536-551): H and the electron-core
// terms contract with D, the two-electron terms are B(D, P) - 1/2 B(P, P) for the symmetric
// bilinear form B(X, Y) = sum X G(Y); D = P gives the energy above.
struct PairDensity {
  double pa[10], pb[10];  // diagonal blocks, tril, off-diagonal entries doubled
  double pab[4][4];       // block (i, j)
};

template <int NI, int NJ>
__device__ void load_pair_density(const double* Pm, int n, int ai, int aj, PairDensity& D) {
#pragma unroll
  for (int k = 0; k < 10; ++k) {
    const int mu = kTriI[k], nu = kTriJ[k];
    const double f = mu == nu ? 1.0 : 2.0;
    D.pa[k] = (mu < NI && nu < NI) ? f * Pm[(size_t)(ai + mu) * n + ai + nu] : 0.0;
    D.pb[k] = (mu < NJ && nu < NJ) ? f * Pm[(size_t)(aj + mu) * n + aj + nu] : 0.0;
  }
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) D.pab[a][b] = (a < NI && b < NJ) ? Pm[(size_t)(ai + a) * n + aj + b] : 0.0;
}

// The nonzero elements of the local tensor (local_tensor): local pair of atom i, of atom j, integral.
__device__ constexpr int kLocP[34] = {0, 0, 0, 0, 0, 1, 1, 1, 1, 1, 2, 2, 2, 2, 2, 5, 5, 5, 5, 5, 9, 9, 9, 9, 9,
                                      3, 3, 4, 4, 6, 6, 7, 7, 8};
__device__ constexpr int kLocQ[34] = {0, 1, 2, 5, 9, 0, 1, 2, 5, 9, 0, 1, 2, 5, 9, 0, 1, 2, 5, 9, 0, 1, 2, 5, 9,
                                      3, 4, 3, 4, 6, 7, 6, 7, 8};
__device__ constexpr int kLocM[34] = {0,  4,  10, 11, 11, 1,  5,  12, 13, 13, 2,  7,  15, 17, 17, 3,  8,
                                      16, 18, 20, 3,  8,  16, 20, 18, 6,  14, 9,  19, 6,  14, 9,  19, 21};

// Density blocks of a pair in its local frame (orbitals s, sigma, pi, pi'; a hydrogen has s only).
struct LocalDensity {
  double a[10], b[10];  // diagonal blocks, tril, plain
  double c[4][4];       // block (i, j)
};

template <int NI, int NJ>
__device__ inline void to_local(const PairDensity& P, const double R[3][3], LocalDensity& out) {
  auto tri = [&](const double (&v)[10], double (&o)[10]) {  // v: off-diagonal entries doubled
    o[0] = v[0];
    double m[3][3];
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int y = 0; y < 3; ++y) m[x][y] = (x == y ? 1.0 : 0.5) * v[tri_index(1 + x, 1 + y)];
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      o[tri_index(1 + x, 0)] = 0.5 * (R[x][0] * v[1] + R[x][1] * v[3] + R[x][2] * v[6]);
      double t[3];
#pragma unroll
      for (int y = 0; y < 3; ++y) t[y] = R[x][0] * m[0][y] + R[x][1] * m[1][y] + R[x][2] * m[2][y];
#pragma unroll
      for (int y = 0; y <= x; ++y) o[tri_index(1 + x, 1 + y)] = t[0] * R[y][0] + t[1] * R[y][1] + t[2] * R[y][2];
    }
  };
  if constexpr (NI == 4) tri(P.pa, out.a);
  if constexpr (NJ == 4) tri(P.pb, out.b);
  if constexpr (NI == 1) out.a[0] = P.pa[0];
  if constexpr (NJ == 1) out.b[0] = P.pb[0];
  double t[4][4];
#pragma unroll
  for (int y = 0; y < NJ; ++y) {
    t[0][y] = P.pab[0][y];
#pragma unroll
    for (int x = 0; x < 3; ++x)
      if (NI == 4) t[1 + x][y] = R[x][0] * P.pab[1][y] + R[x][1] * P.pab[2][y] + R[x][2] * P.pab[3][y];
  }
#pragma unroll
  for (int x = 0; x < NI; ++x) {
    out.c[x][0] = t[x][0];
#pragma unroll
    for (int y = 0; y < 3; ++y)
      if (NJ == 4) out.c[x][1 + y] = R[y][0] * t[x][1] + R[y][1] * t[x][2] + R[y][2] * t[x][3];
  }
}

// The change of a local block element when the axis turns towards local orbital K (2: pi, 3: pi'):
// d sigma = orbital K, d (orbital K) = - sigma, on the first (second) index where the atom has p orbitals.
template <int K>
__device__ inline double turn_tri(const double (&m)[10], int x, int y) {
  double d = 0.0;
  if (x == 1) d += m[tri_index(K, y)];
  if (x == K) d -= m[tri_index(1, y)];
  if (y == 1) d += m[tri_index(x, K)];
  if (y == K) d -= m[tri_index(x, 1)];
  return d;
}
template <int K, int NI, int NJ>
__device__ inline double turn_ab(const double (&m)[4][4], int x, int y) {
  double d = 0.0;
  if (NI == 4 && x == 1) d += m[K][y];
  if (NI == 4 && x == K) d -= m[1][y];
  if (NJ == 4 && y == 1) d += m[x][K];
  if (NJ == 4 && y == K) d -= m[x][1];
  return d;
}

// Two-electron (and, with ELCORE, electron-core) potential of the local density M, contracted with
// the change of the local density X as the axis turns towards pi (t[0]) and pi' (t[1]).
template <int KIND, bool ELCORE>
__device__ inline void axis_torque(const Dual* ri, const LocalDensity& M, const LocalDensity& X, double ti, double tj,
                                   double (&t)[2]) {
  constexpr int NJ = KIND == XX ? 4 : 1;
  constexpr int NE = KIND == XX ? 34 : 5;
  double ja[10], jb[10], K[4][4];
#pragma unroll
  for (int k = 0; k < 10; ++k) ja[k] = jb[k] = 0.0;
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y) K[x][y] = 0.0;
  constexpr int xhP[5] = {0, 1, 2, 5, 9}, xhM[5] = {0, 1, 2, 3, 3};
#pragma unroll
  for (int q = 0; q < NE; ++q) {
    const int p = KIND == XX ? kLocP[q] : xhP[q], o = KIND == XX ? kLocQ[q] : 0;
    const double w = ri[KIND == XX ? kLocM[q] : xhM[q]].v;
    const int mu = kTriI[p], nu = kTriJ[p], la = kTriI[o], si = kTriJ[o];
    ja[p] += (la == si ? w : 2.0 * w) * M.b[o];
    if (ELCORE && o == 0) ja[p] -= tj * w;
    if (KIND == XX) {
      jb[o] += (mu == nu ? w : 2.0 * w) * M.a[p];
      if (ELCORE && p == 0) jb[o] -= ti * w;
    }
    K[mu][la] += w * M.c[nu][si];
    if (mu != nu) K[nu][la] += w * M.c[mu][si];
    if (la != si) K[mu][si] += w * M.c[nu][la];
    if (mu != nu && la != si) K[nu][si] += w * M.c[mu][la];
  }
#pragma unroll
  for (int p = 1; p < 10; ++p) {
    const int mu = kTriI[p], nu = kTriJ[p];
    const double f = mu == nu ? 1.0 : 2.0;
    t[0] += f * ja[p] * turn_tri<2>(X.a, mu, nu);
    t[1] += f * ja[p] * turn_tri<3>(X.a, mu, nu);
    if (KIND == XX) {
      t[0] += f * jb[p] * turn_tri<2>(X.b, mu, nu);
      t[1] += f * jb[p] * turn_tri<3>(X.b, mu, nu);
    }
  }
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < NJ; ++y) {
      t[0] -= K[x][y] * turn_ab<2, 4, NJ>(X.c, x, y);
      t[1] -= K[x][y] * turn_ab<3, 4, NJ>(X.c, x, y);
    }
}

// dE_pair/dR (R = r_j - r_i, Angstrom) of the pair energy above at fixed densities, in closed form.  In the
// frame of the pair axis the energy is sum_m c_m ri_m(r) (22 local integrals, c_m bilinear in the local
// densities) + sum_m o_m S_m(r) (5 overlaps) + core repulsion(r): the derivative along the axis takes each of those functions of r once with its derivative (Dual), and the
// two derivatives across the axis are the turns of the local densities under the local potential.
// Inside the antipodal fallback cone a frame is constant (the reference's autograd gives it no
// derivative), which drops that frame's part across the axis; the overlaps keep their B-integral branch.
// Bound: FP64 VALU and its latencies (about 64 inverse roots and 8 exponentials per heavy-heavy pair),
// one wave per SIMD in the heavy-heavy kernel (256 VGPRs and as many accumulation registers).  Against
// 12 displaced energies per pair (4th-order differences, each rotating all 100 integrals) on 512
// alkanes of 2-30 carbons: heavy-heavy 1156 -> 42 us, heavy-H 393 -> 35 us, H-H 187 -> 24 us; one
// ethane 311 -> 17 us.  The differences agree with it to 2e-10 of the force norm, their rounding.
template <int KIND, bool XL>
__device__ inline void pair_gradient(int method, const double (&R0)[3], const double* pi, const double* pj,
                                     const PairDensity& P, const PairDensity& D, double (&G)[3]) {
  constexpr int NI = KIND == HH ? 1 : 4;
  constexpr int NJ = KIND == XX ? 4 : 1;
  const PairGeom g = geom_from_vector(R0[0], R0[1], R0[2]);
  const Dual r = {g.r, 1.0};
  const double ti = pi[PAR_TORE], tj = pj[PAR_TORE];
  double along = 0.0;                  // dE/dr, eV/bohr
  double across[3] = {0.0, 0.0, 0.0};  // dE/d(unit vector i -> j), before projection off the axis
  // resonance: sum 2 D_ab H_ab
  if (g.r <= kOverlapCut) {
    const bool fixed = quat_flips(g.x[0]);
    double Rp[3][3];
    quat_frame(g.x[0], g.x[1], g.x[2], Rp, fixed ? 2 : 1);
    const double u[3] = {Rp[0][0], Rp[0][1], Rp[0][2]};
    Dual S[5];
    overlap_local<Dual, KIND>(jcall_of((int)pi[PAR_QN], (int)pj[PAR_QN]), r, pi[PAR_ZS], pi[PAR_ZP], pj[PAR_ZS],
                              pj[PAR_ZP], NI == 4, S);
    along += D.pab[0][0] * (pi[PAR_BS] + pj[PAR_BS]) * S[0].d;
    if constexpr (NI == 4) {
      const double bps = pi[PAR_BP] + pj[PAR_BS];
      along += bps * (D.pab[1][0] * u[0] + D.pab[2][0] * u[1] + D.pab[3][0] * u[2]) * S[1].d;
      if (!fixed)
#pragma unroll
        for (int m = 0; m < 3; ++m) across[m] += bps * S[1].v * D.pab[1 + m][0];
    }
    if constexpr (NJ == 4) {
      const double bsp = pi[PAR_BS] + pj[PAR_BP], bpp = pi[PAR_BP] + pj[PAR_BP];
      along -= bsp * (D.pab[0][1] * u[0] + D.pab[0][2] * u[1] + D.pab[0][3] * u[2]) * S[2].d;
      double du[3], duu = 0.0;
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        du[m] = 0.0;
#pragma unroll
        for (int k = 0; k < 3; ++k) du[m] += (D.pab[1 + m][1 + k] + D.pab[1 + k][1 + m]) * u[k];
        duu += 0.5 * du[m] * u[m];
      }
      const double tr = D.pab[1][1] + D.pab[2][2] + D.pab[3][3];
      along += bpp * ((tr - duu) * S[4].d - duu * S[3].d);
      if (!fixed)
#pragma unroll
        for (int m = 0; m < 3; ++m)
          across[m] -= bsp * S[2].v * D.pab[0][1 + m] + bpp * (S[3].v + S[4].v) * du[m];
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // the overlaps' registers are free again below
  // two-electron, electron-core and core-core terms
  Dual gam;
  if constexpr (KIND == HH) {
    const double rho = pi[PAR_RHO0] + pj[PAR_RHO0];
    gam = quot_root(kEV, r * r + rho * rho);
    const double cw = XL ? D.pa[0] * P.pb[0] + P.pa[0] * D.pb[0] - P.pa[0] * P.pb[0] : P.pa[0] * P.pb[0];
    const double xw = XL ? D.pab[0][0] - 0.5 * P.pab[0][0] : 0.5 * P.pab[0][0];
    along += (cw - tj * D.pa[0] - ti * D.pb[0] - xw * P.pab[0][0]) * gam.d;
  } else {
    const bool fixed = quat_flips(-g.x[0]);
    double R[3][3];
    quat_frame(-g.x[0], -g.x[1], -g.x[2], R, fixed ? 2 : 1);
    LocalDensity Pl, Dl;
    to_local<NI, NJ>(P, R, Pl);
    if constexpr (XL) to_local<NI, NJ>(D, R, Dl);
    Dual ri[22];
    if constexpr (KIND == XX)
      local_xx<Dual>(r, pi[PAR_DD], pj[PAR_DD], pi[PAR_QQ], pj[PAR_QQ], pi[PAR_RHO0], pj[PAR_RHO0], pi[PAR_RHO1],
                     pj[PAR_RHO1], pi[PAR_RHO2], pj[PAR_RHO2], ri);
    else
      local_xh<Dual>(r, pi[PAR_DD], pi[PAR_QQ], pi[PAR_RHO0], pi[PAR_RHO1], pi[PAR_RHO2], pj[PAR_RHO0], ri);
    gam = ri[0];
    const LocalDensity& E = XL ? Dl : Pl;
    constexpr int NE = KIND == XX ? 34 : 5;
    constexpr int xhP[5] = {0, 1, 2, 5, 9}, xhM[5] = {0, 1, 2, 3, 3};
    auto xw = [&](int x, int y) { return XL ? Dl.c[x][y] - 0.5 * Pl.c[x][y] : 0.5 * Pl.c[x][y]; };
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      const int p = KIND == XX ? kLocP[q] : xhP[q], o = KIND == XX ? kLocQ[q] : 0;
      const int mu = kTriI[p], nu = kTriJ[p], la = kTriI[o], si = kTriJ[o];
      double c = XL ? Dl.a[p] * Pl.b[o] + Pl.a[p] * (Dl.b[o] - Pl.b[o]) : Pl.a[p] * Pl.b[o];
      if (o == 0) c -= tj * E.a[p];
      if (mu != nu) c *= 2.0;
      double cb = 0.0;
      if (p == 0) cb = ti * E.b[o];
      if (la != si) {
        c *= 2.0;
        cb *= 2.0;
      }
      c -= cb;
      c -= xw(mu, la) * Pl.c[nu][si];
      if (mu != nu) c -= xw(nu, la) * Pl.c[mu][si];
      if (la != si) c -= xw(mu, si) * Pl.c[nu][la];
      if (mu != nu && la != si) c -= xw(nu, si) * Pl.c[mu][la];
      along += c * ri[KIND == XX ? kLocM[q] : xhM[q]].d;
    }
    __builtin_amdgcn_sched_barrier(0);
    if (!fixed) {
      double t[2] = {0.0, 0.0};
      axis_torque<KIND, true>(ri, Pl, E, ti, tj, t);
      if constexpr (XL) {  // the potential of D - P on the turn of P
#pragma unroll
        for (int k = 0; k < 10; ++k) {
          Dl.a[k] -= Pl.a[k];
          if (NJ == 4 || k == 0) Dl.b[k] -= Pl.b[k];
        }
#pragma unroll
        for (int x = 0; x < NI; ++x)
#pragma unroll
          for (int y = 0; y < NJ; ++y) Dl.c[x][y] -= Pl.c[x][y];
        axis_torque<KIND, false>(ri, Dl, Pl, ti, tj, t);
      }
      // the frame's sigma points from j to i: turning it towards pi moves the unit vector i -> j by -pi
#pragma unroll
      for (int m = 0; m < 3; ++m) across[m] -= t[0] * R[1][m] + t[1] * R[2][m];
    }
  }
  along += core_repulsion<Dual>(method, (int)pi[PAR_Z], (int)pj[PAR_Z], r, gam, pi, pj).d;
  const double off = across[0] * g.x[0] + across[1] * g.x[1] + across[2] * g.x[2];
  const double rd = 1.0 / (g.r * kA0);
#pragma unroll
  for (int m = 0; m < 3; ++m) G[m] = along * (1.0 / kA0) * g.x[m] + rd * (across[m] - off * g.x[m]);
}

// Forces: +dE/dR on atom i, -dE/dR on atom j, reduced per tile.
// XL: Dm is the density contracted with H (the XL-BOMD D), P the propagated field.
template <int KIND, bool XL>
__device__ __forceinline__ void force_tile(const pyseqm_layout_t& L, int method, int tile,
                                           const double* __restrict__ coords, const double* __restrict__ par,
                                           const double* __restrict__ P, const double* __restrict__ Dm,
                                           double* __restrict__ part) {
  const int lane = threadIdx.x;
  const Tile t = load_tile(L.tiles, tile);
  int i, j;
  const bool valid = lane_pair(t, lane, i, j);
  double rowv[3] = {0.0, 0.0, 0.0}, colv[3] = {0.0, 0.0, 0.0};
  if (valid) {
    const double* pi = par + (size_t)i * PYSEQM_NPAR;
    const double* pj = par + (size_t)j * PYSEQM_NPAR;
    const long long mo = L.mol_mat_off[t.mol];
    const int n = L.mol_norb[t.mol];
    const int ai = L.atom_ao[i], aj = L.atom_ao[j];
    constexpr int NI = KIND == HH ? 1 : 4;
    constexpr int NJ = KIND == XX ? 4 : 1;
    PairDensity Pd, Dd;
    load_pair_density<NI, NJ>(P + mo, n, ai, aj, Pd);
    if constexpr (XL) load_pair_density<NI, NJ>(Dm + mo, n, ai, aj, Dd);
    const double R0[3] = {coords[3 * j] - coords[3 * i], coords[3 * j + 1] - coords[3 * i + 1],
                          coords[3 * j + 2] - coords[3 * i + 2]};
    pair_gradient<KIND, XL>(method, R0, pi, pj, Pd, XL ? Dd : Pd, rowv);
#pragma unroll
    for (int x = 0; x < 3; ++x) colv[x] = -rowv[x];
  }
  write_partials(part, tile, lane, rowv, colv);
}

template <int KIND, bool XL>
__global__ __launch_bounds__(64) void k_pair_forces(pyseqm_layout_t L, int method, int tile_base,
                                                    const double* __restrict__ coords,
                                                    const double* __restrict__ par, const double* __restrict__ P,
                                                    const double* __restrict__ Dm, double* __restrict__ part) {
  for_tile<KIND>(L, tile_base, [&](auto kind, int tile) {
    force_tile<decltype(kind)::value, XL>(L, method, tile, coords, par, P, Dm, part);
  });
}

template <int G>
__global__ __launch_bounds__(256) void k_atom_forces(pyseqm_layout_t L, const double* __restrict__ part,
                                                     double* __restrict__ F) {
  const int a = blockIdx.x * (256 / G) + threadIdx.x / G;
  const int lane = threadIdx.x % G;
  if (a >= L.natoms) return;  // uniform over the lane group
  double f[3];
  gather_slots<G>(part, L.csr_idx, L.csr_off[a], L.csr_off[a + 1], lane, f);
  if (lane < 3) F[3 * a + lane] = lane == 0 ? f[0] : (lane == 1 ? f[1] : f[2]);
}

// ------------------------------------------------- energy gradient w.r.t. atom parameters
// At a converged closed-shell SCF density the energy is stationary in P, so dE/dtheta is the
// derivative at fixed P: the gradient the reference's autograd returns through H, the integrals and
// the core repulsion when the SCF density is detached (scf_backward = 0, scf_loop.py:1996-2031;
// learned parameters re-packed per call, basics.py:781-789).  A pair's energy depends on the inputs of
// its two atoms through few quantities per atom (kPV below), and its derivatives in them are closed:
//   * the multipoles dd, qq, rho0, rho1, rho2: the two-electron and electron-core terms are
//     sum_m c_m ri_m, with c_m bilinear in the densities rotated to the pair's frame and every ri_m a
//     sum of inverse roots, which are differentiated one by one (charge_terms);
//   * rho0 once more through the core repulsion's (ss|ss);
//   * the exponents, through the 5 overlaps (Dual, on the B-integral branch of the pair);
//   * the resonance integrals, which enter linearly, alpha and the Gaussians.
// k_param_jacobian has the derivative of each atom's multipoles in its inputs (4th-order differences of
// derive_atom, whose secant iterations have no short closed form), and k_param_gather joins the two.
// U_ss, U_pp and g_sp reach the one-center terms only, which k_param_onecenter differentiates.
// One pass over the pairs with 23 values per side, where displaced energies took 4 x 2 x 21 pair energies
// in 5 passes: on 32 alkanes of 1-8 carbons 6760 -> 37 us (+ 42 us
// for the Jacobian).
constexpr int kPV = 23;  // dd qq rho0 rho1 rho2 | core repulsion's rho0 | zs zp bs bp | alpha | 12 Gaussian
enum { PV_DD = 0, PV_QQ, PV_R0, PV_R1, PV_R2, PV_REP, PV_ZS, PV_ZP, PV_BS, PV_BP, PV_ALPHA, PV_GAUSS };
constexpr int kJacSlots = 6;
__device__ constexpr int kJacParam[kJacSlots] = {PAR_ZS, PAR_ZP, PAR_GSS, PAR_GPP, PAR_GP2, PAR_HSP};
__device__ constexpr int kJacOut[5] = {PAR_DD, PAR_QQ, PAR_RHO0, PAR_RHO1, PAR_RHO2};

// jac[(a * 6 + k) * 5 + y]: d(multipole kJacOut[y])/d(input kJacParam[k]) of atom a, by 4th-order central
// differences with step hrel * max(|value|, 0.1).  One thread per (atom, input).
__global__ void k_param_jacobian(pyseqm_layout_t L, const double* __restrict__ par, double hrel,
                                 double* __restrict__ jac) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int a = t / kJacSlots, k = t - a * kJacSlots;
  if (a >= L.natoms) return;
  const double* src = par + (size_t)a * PYSEQM_NPAR;
  const int slot = kJacParam[k], Z = L.atom_Z[a];
  const double h = hrel * fmax(fabs(src[slot]), 0.1);
  double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  for (int s = -2; s <= 2; ++s) {
    if (s == 0) continue;
    double q[PYSEQM_NPAR];
    for (int i = 0; i < PYSEQM_NPAR; ++i) q[i] = src[i];
    q[slot] = src[slot] + s * h;
    derive_atom(q, Z);
    const double w = s == -2 ? 1.0 : (s == -1 ? -8.0 : (s == 1 ? 8.0 : -1.0));
    for (int y = 0; y < 5; ++y) acc[y] += w * q[kJacOut[y]];
  }
  for (int y = 0; y < 5; ++y) jac[(size_t)t * 5 + y] = acc[y] / (12.0 * h);
}

// d(sum_m c_m ri_m)/d(multipoles) of a heavy-heavy pair (local_xx): ga for atom i, gb for atom j, in the
// order dd, qq, rho0, rho1, rho2.  Every term is A / sqrt(u^2 + v^2 + (rho_a + rho_b)^2) with u, v
// linear in r, da, db, qa, qb; g = -A / root^3 times u, v or the rho sum gives its derivatives.
struct ChargeTerms {
  double da, db, qa, qb;        // the charge offsets (qa, qb: local_xx's qa1, qb1)
  double ra[3], rb[3];          // rho0, rho1, rho2
  double gda, gdb, gqa, gqb;    // derivatives in the offsets
  double gra[3], grb[3];        // derivatives in the rhos
  // A / sqrt((r + s_da da + ..)^2 + (t_da da + ..)^2 + (rho_I + rho_J)^2)
  template <int I, int J>
  __device__ inline void term(double r, double A, double sda, double sdb, double sqa, double sqb, double tda = 0.0,
                              double tdb = 0.0, double tqa = 0.0, double tqb = 0.0) {
    const double u = r + sda * da + sdb * db + sqa * qa + sqb * qb;
    const double v = tda * da + tdb * db + tqa * qa + tqb * qb;
    const double w = ra[I] + rb[J];
    const double q = rsq_nr(u * u + v * v + w * w);
    const double g = -A * (q * q * q);
    gda += g * (sda * u + tda * v);
    gdb += g * (sdb * u + tdb * v);
    gqa += g * (sqa * u + tqa * v);
    gqb += g * (sqb * u + tqb * v);
    gra[I] += g * w;
    grb[J] += g * w;
  }
};

__device__ inline void charge_terms_xx(double r, const double (&c)[22], ChargeTerms& t) {
  const double e1 = kEV * 0.5, e2 = kEV * 0.25, e3 = kEV * 0.125, e4 = kEV * 0.0625;
  const double ee = c[0] + c[2] + c[3] + c[10] + c[11] + c[15] + c[16] + c[17] + c[18] + c[20];
  t.term<0, 0>(r, kEV * ee, 0, 0, 0, 0);
  const double dze = -(c[1] + c[12] + c[13]);
  t.term<1, 0>(r, -e1 * dze, 1, 0, 0, 0);
  t.term<1, 0>(r, e1 * dze, -1, 0, 0, 0);
  const double edz = -(c[4] + c[7] + c[8]);
  t.term<0, 1>(r, -e1 * edz, 0, -1, 0, 0);
  t.term<0, 1>(r, e1 * edz, 0, 1, 0, 0);
  __builtin_amdgcn_sched_barrier(0);
  const double qzze = c[2] + c[15] + c[17], qxxe = c[3] + c[16] + c[18] + c[20];
  t.term<2, 0>(r, e2 * qzze, 0, 0, -2, 0);
  t.term<2, 0>(r, e2 * qzze, 0, 0, 2, 0);
  t.term<2, 0>(r, -e1 * (qzze + qxxe), 0, 0, 0, 0);
  t.term<2, 0>(r, e1 * qxxe, 0, 0, 0, 0, 0, 0, 2, 0);
  const double eqzz = c[10] + c[15] + c[16], eqxx = c[11] + c[17] + c[18] + c[20];
  t.term<0, 2>(r, e2 * eqzz, 0, 0, 0, -2);
  t.term<0, 2>(r, e2 * eqzz, 0, 0, 0, 2);
  t.term<0, 2>(r, -e1 * (eqzz + eqxx), 0, 0, 0, 0);
  t.term<0, 2>(r, e1 * eqxx, 0, 0, 0, 0, 0, 0, 0, 2);
  // dipole-dipole
  __builtin_amdgcn_sched_barrier(0);
  t.term<1, 1>(r, e2 * c[5], 1, -1, 0, 0);
  t.term<1, 1>(r, e2 * c[5], -1, 1, 0, 0);
  t.term<1, 1>(r, -e2 * c[5], -1, -1, 0, 0);
  t.term<1, 1>(r, -e2 * c[5], 1, 1, 0, 0);
  t.term<1, 1>(r, e1 * c[6], 0, 0, 0, 0, 1, -1, 0, 0);
  t.term<1, 1>(r, -e1 * c[6], 0, 0, 0, 0, 1, 1, 0, 0);
  // quadrupole (i) - dipole (j)
  __builtin_amdgcn_sched_barrier(0);
  const double c78 = c[7] + c[8];
  t.term<2, 1>(r, -e2 * c78, 0, -1, 0, 0);
  t.term<2, 1>(r, e2 * c78, 0, 1, 0, 0);
  t.term<2, 1>(r, e3 * c[7], 0, -1, 2, 0);
  t.term<2, 1>(r, -e3 * c[7], 0, 1, 2, 0);
  t.term<2, 1>(r, e3 * c[7], 0, -1, -2, 0);
  t.term<2, 1>(r, -e3 * c[7], 0, 1, -2, 0);
  t.term<2, 1>(r, e2 * c[8], 0, -1, 0, 0, 0, 0, 2, 0);
  t.term<2, 1>(r, -e2 * c[8], 0, 1, 0, 0, 0, 0, 2, 0);
  __builtin_amdgcn_sched_barrier(0);
  t.term<2, 1>(r, e2 * c[9], 0, 0, 1, 0, 0, -1, 1, 0);
  t.term<2, 1>(r, -e2 * c[9], 0, 0, -1, 0, 0, -1, 1, 0);
  t.term<2, 1>(r, -e2 * c[9], 0, 0, 1, 0, 0, 1, 1, 0);
  t.term<2, 1>(r, e2 * c[9], 0, 0, -1, 0, 0, 1, 1, 0);
  // dipole (i) - quadrupole (j)
  __builtin_amdgcn_sched_barrier(0);
  const double c1213 = c[12] + c[13];
  t.term<1, 2>(r, -e2 * c1213, 1, 0, 0, 0);
  t.term<1, 2>(r, e2 * c1213, -1, 0, 0, 0);
  t.term<1, 2>(r, e3 * c[12], 1, 0, 0, -2);
  t.term<1, 2>(r, -e3 * c[12], -1, 0, 0, -2);
  t.term<1, 2>(r, e3 * c[12], 1, 0, 0, 2);
  t.term<1, 2>(r, -e3 * c[12], -1, 0, 0, 2);
  t.term<1, 2>(r, e2 * c[13], 1, 0, 0, 0, 0, 0, 0, 2);
  t.term<1, 2>(r, -e2 * c[13], -1, 0, 0, 0, 0, 0, 0, 2);
  __builtin_amdgcn_sched_barrier(0);
  t.term<1, 2>(r, e2 * c[14], 0, 0, 0, -1, 1, 0, 0, -1);
  t.term<1, 2>(r, -e2 * c[14], 0, 0, 0, 1, 1, 0, 0, -1);
  t.term<1, 2>(r, -e2 * c[14], 0, 0, 0, -1, 1, 0, 0, 1);
  t.term<1, 2>(r, e2 * c[14], 0, 0, 0, 1, 1, 0, 0, 1);
  // quadrupole-quadrupole
  __builtin_amdgcn_sched_barrier(0);
  t.term<2, 2>(r, e4 * c[15], 0, 0, 2, -2);
  t.term<2, 2>(r, e4 * c[15], 0, 0, 2, 2);
  t.term<2, 2>(r, e4 * c[15], 0, 0, -2, -2);
  t.term<2, 2>(r, e4 * c[15], 0, 0, -2, 2);
  t.term<2, 2>(r, -e3 * (c[15] + c[16]), 0, 0, 0, -2);
  t.term<2, 2>(r, -e3 * (c[15] + c[16]), 0, 0, 0, 2);
  t.term<2, 2>(r, -e3 * (c[15] + c[17]), 0, 0, 2, 0);
  t.term<2, 2>(r, -e3 * (c[15] + c[17]), 0, 0, -2, 0);
  __builtin_amdgcn_sched_barrier(0);
  t.term<2, 2>(r, e2 * (c[15] + c[16] + c[17] + c[18] + c[20]), 0, 0, 0, 0);
  t.term<2, 2>(r, -e2 * (c[16] + c[18] + c[20]), 0, 0, 0, 0, 0, 0, 2, 0);
  t.term<2, 2>(r, -e2 * (c[17] + c[18] + c[20]), 0, 0, 0, 0, 0, 0, 0, 2);
  t.term<2, 2>(r, e3 * c[16], 0, 0, 0, -2, 0, 0, 2, 0);
  t.term<2, 2>(r, e3 * c[16], 0, 0, 0, 2, 0, 0, 2, 0);
  t.term<2, 2>(r, e3 * c[17], 0, 0, 2, 0, 0, 0, 0, 2);
  t.term<2, 2>(r, e3 * c[17], 0, 0, -2, 0, 0, 0, 0, 2);
  __builtin_amdgcn_sched_barrier(0);
  const double cxx = c[18] + 0.5 * c[21], cxy = c[20] - 0.5 * c[21];
  t.term<2, 2>(r, e3 * cxx, 0, 0, 0, 0, 0, 0, 2, -2);
  t.term<2, 2>(r, e3 * cxx, 0, 0, 0, 0, 0, 0, 2, 2);
  {  // e2 cxy / sqrt(r^2 + (2 qa)^2 + (2 qb)^2 + ..): two offsets across the axis
    const double w = t.ra[2] + t.rb[2];
    const double q = rsq_nr(r * r + 4.0 * t.qa * t.qa + 4.0 * t.qb * t.qb + w * w);
    const double g = -e2 * cxy * (q * q * q);
    t.gqa += 4.0 * g * t.qa;
    t.gqb += 4.0 * g * t.qb;
    t.gra[2] += g * w;
    t.grb[2] += g * w;
  }
  __builtin_amdgcn_sched_barrier(0);
  t.term<2, 2>(r, e3 * c[19], 0, 0, 1, -1, 0, 0, 1, -1);
  t.term<2, 2>(r, -e3 * c[19], 0, 0, 1, 1, 0, 0, 1, -1);
  t.term<2, 2>(r, -e3 * c[19], 0, 0, -1, -1, 0, 0, 1, -1);
  t.term<2, 2>(r, e3 * c[19], 0, 0, -1, 1, 0, 0, 1, -1);
  t.term<2, 2>(r, -e3 * c[19], 0, 0, 1, -1, 0, 0, 1, 1);
  t.term<2, 2>(r, e3 * c[19], 0, 0, 1, 1, 0, 0, 1, 1);
  t.term<2, 2>(r, e3 * c[19], 0, 0, -1, -1, 0, 0, 1, 1);
  t.term<2, 2>(r, -e3 * c[19], 0, 0, -1, 1, 0, 0, 1, 1);
}

// the same for a heavy-H pair (local_xh)
__device__ inline void charge_terms_xh(double r, const double (&c)[4], ChargeTerms& t) {
  const double e1 = kEV * 0.5, e2 = kEV * 0.25;
  t.term<0, 0>(r, kEV * (c[0] + c[2] + c[3]), 0, 0, 0, 0);
  t.term<1, 0>(r, e1 * c[1], 1, 0, 0, 0);
  t.term<1, 0>(r, -e1 * c[1], -1, 0, 0, 0);
  t.term<2, 0>(r, e2 * c[2], 0, 0, 2, 0);
  t.term<2, 0>(r, e2 * c[2], 0, 0, -2, 0);
  t.term<2, 0>(r, -e1 * (c[2] + c[3]), 0, 0, 0, 0);
  t.term<2, 0>(r, e1 * c[3], 0, 0, 0, 0, 0, 0, 2, 0);
}

// A pair's derivatives in the quantities of atom i (row partial) and of atom j (column partial), MODE 0
// of Eelec(P) and of the core repulsion, MODE 2 of sum Y F(P) for a symmetric Y (no core repulsion).
template <int KIND, int MODE>
__global__ __launch_bounds__(64) void k_pair_param_grad(pyseqm_layout_t L, int method, int tile_base,
                                                        const double* __restrict__ coords,
                                                        const double* __restrict__ par, const double* __restrict__ P,
                                                        const double* __restrict__ Y, double* __restrict__ part) {
  const int tile = tile_base + xcd_run(blockIdx.x, gridDim.x);
  const int lane = threadIdx.x;
  const Tile t = load_tile(L.tiles, tile);
  int i, j;
  const bool valid = lane_pair(t, lane, i, j);
  // lanes without a pair take the tile's first row and column (both exist) and add zeros below
  if (!valid) {
    i = t.row0;
    j = t.col0 + t.ncol - 1;
  }
  const double* pi = par + (size_t)i * PYSEQM_NPAR;
  const double* pj = par + (size_t)j * PYSEQM_NPAR;
  const int r8 = lane >> 3, c8 = lane & 7;
  double* prow = part + ((size_t)tile * 16 + r8) * kPV;
  double* pcol = part + ((size_t)tile * 16 + 8 + c8) * kPV;
  // value k of the tile's row and column partials, written as soon as it is known (every lane active)
  auto put = [&](int k, double row, double col) {
    const double rs = row8(valid ? row : 0.0), cs = col8(valid ? col : 0.0);
    if (c8 == 0) prow[k] = rs;
    if (r8 == 0) pcol[k] = cs;
  };
  const long long mo = L.mol_mat_off[t.mol];
  const int n = L.mol_norb[t.mol];
  constexpr int NI = KIND == HH ? 1 : 4;
  constexpr int NJ = KIND == XX ? 4 : 1;
  PairDensity Pd, Yd;
  load_pair_density<NI, NJ>(P + mo, n, L.atom_ao[i], L.atom_ao[j], Pd);
  if constexpr (MODE == 2) load_pair_density<NI, NJ>(Y + mo, n, L.atom_ao[i], L.atom_ao[j], Yd);
  const PairDensity& D = MODE == 2 ? Yd : Pd;  // contracted with H and the electron-core terms
  const PairGeom g = pair_geom(coords, i, j);
  const double ti = pi[PAR_TORE], tj = pj[PAR_TORE];
  {
    double zr[4] = {0.0, 0.0, 0.0, 0.0}, zc[4] = {0.0, 0.0, 0.0, 0.0};
    // overlaps: exponents and resonance integrals
    if (g.r <= kOverlapCut) {
      double Rp[3][3];
      quat_frame(g.x[0], g.x[1], g.x[2], Rp, quat_flips(g.x[0]) ? 2 : 1);
      const double d0 = D.pab[0][0];
      double d1 = 0.0, d2 = 0.0, duu = 0.0, tr = 0.0;
      if constexpr (NI == 4) d1 = D.pab[1][0] * Rp[0][0] + D.pab[2][0] * Rp[0][1] + D.pab[3][0] * Rp[0][2];
      if constexpr (NJ == 4) {
        d2 = -(D.pab[0][1] * Rp[0][0] + D.pab[0][2] * Rp[0][1] + D.pab[0][3] * Rp[0][2]);
#pragma unroll
        for (int m = 0; m < 3; ++m) {
          tr += D.pab[1 + m][1 + m];
#pragma unroll
          for (int k = 0; k < 3; ++k) duu += Rp[0][m] * D.pab[1 + m][1 + k] * Rp[0][k];
        }
      }
      const int jc = jcall_of((int)pi[PAR_QN], (int)pj[PAR_QN]);
      const double bss = pi[PAR_BS] + pj[PAR_BS], bps = pi[PAR_BP] + pj[PAR_BS], bsp = pi[PAR_BS] + pj[PAR_BP],
                   bpp = pi[PAR_BP] + pj[PAR_BP];
      // each overlap depends on one exponent per side, so one pass per side serves s and p
#pragma unroll 1
      for (int side = 0; side < 2; ++side) {
        const double sa = side == 0 ? 1.0 : 0.0, sb = 1.0 - sa;
        Dual S[5];
        overlap_local<Dual, KIND>(jc, g.r, Dual{pi[PAR_ZS], sa}, Dual{pi[PAR_ZP], sa}, Dual{pj[PAR_ZS], sb},
                                  Dual{pj[PAR_ZP], sb}, NI == 4, S);
        const double ss = bss * d0 * S[0].d, ps = bps * d1 * S[1].d, sp = bsp * d2 * S[2].d;
        const double pp = bpp * ((tr - duu) * S[4].d - duu * S[3].d);
        const double vss = d0 * S[0].v, vps = d1 * S[1].v, vsp = d2 * S[2].v;
        const double vpp = (tr - duu) * S[4].v - duu * S[3].v;
        if (side == 0) {
          zr[0] = ss + sp;
          zr[1] = ps + pp;
          zr[2] = vss + vsp;
          zr[3] = vps + vpp;
        } else {
          zc[0] = ss + ps;
          zc[1] = sp + pp;
          zc[2] = vss + vps;
          zc[3] = vsp + vpp;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) put(PV_ZS + k, zr[k], zc[k]);
  }
  __builtin_amdgcn_sched_barrier(0);
  {
    // two-electron and electron-core terms: the multipoles
    ChargeTerms q = {pi[PAR_DD], pj[PAR_DD], pi[PAR_QQ], pj[PAR_QQ],
                     {pi[PAR_RHO0], pi[PAR_RHO1], pi[PAR_RHO2]}, {pj[PAR_RHO0], pj[PAR_RHO1], pj[PAR_RHO2]},
                     0.0, 0.0, 0.0, 0.0, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
    if constexpr (KIND == HH) {
      const double cw = MODE == 2 ? D.pa[0] * Pd.pb[0] + Pd.pa[0] * D.pb[0] : Pd.pa[0] * Pd.pb[0];
      const double xw = MODE == 2 ? D.pab[0][0] : 0.5 * Pd.pab[0][0];
      q.term<0, 0>(g.r, kEV * (cw - tj * D.pa[0] - ti * D.pb[0] - xw * Pd.pab[0][0]), 0, 0, 0, 0);
    } else {
      double R[3][3];
      quat_frame(-g.x[0], -g.x[1], -g.x[2], R, quat_flips(-g.x[0]) ? 2 : 1);
      LocalDensity Pl, Yl;
      to_local<NI, NJ>(Pd, R, Pl);
      if constexpr (MODE == 2) to_local<NI, NJ>(Yd, R, Yl);
      const LocalDensity& E = MODE == 2 ? Yl : Pl;
      constexpr int NM = KIND == XX ? 22 : 4, NE = KIND == XX ? 34 : 5;
      constexpr int xhP[5] = {0, 1, 2, 5, 9}, xhM[5] = {0, 1, 2, 3, 3};
      const double xf = MODE == 2 ? 1.0 : 0.5;
      double cm[NM];
#pragma unroll
      for (int k = 0; k < NM; ++k) cm[k] = 0.0;
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int p = KIND == XX ? kLocP[e] : xhP[e], o = KIND == XX ? kLocQ[e] : 0;
        const int mu = kTriI[p], nu = kTriJ[p], la = kTriI[o], si = kTriJ[o];
        const double fp = mu == nu ? 1.0 : 2.0, fo = la == si ? 1.0 : 2.0;
        double c = MODE == 2 ? Yl.a[p] * Pl.b[o] + Pl.a[p] * Yl.b[o] : Pl.a[p] * Pl.b[o];
        c *= fp * fo;
        if (o == 0) c -= tj * fp * E.a[p];
        if (p == 0) c -= ti * fo * E.b[o];
        double x = E.c[mu][la] * Pl.c[nu][si];
        if (mu != nu) x += E.c[nu][la] * Pl.c[mu][si];
        if (la != si) x += E.c[mu][si] * Pl.c[nu][la];
        if (mu != nu && la != si) x += E.c[nu][si] * Pl.c[mu][la];
        cm[KIND == XX ? kLocM[e] : xhM[e]] += c - xf * x;
      }
      if constexpr (KIND == XX)
        charge_terms_xx(g.r, cm, q);
      else
        charge_terms_xh(g.r, cm, q);
    }
    put(PV_DD, q.gda, q.gdb);
    put(PV_QQ, q.gqa, q.gqb);
#pragma unroll
    for (int k = 0; k < 3; ++k) put(PV_R0 + k, q.gra[k], q.grb[k]);
  }
  __builtin_amdgcn_sched_barrier(0);
  // core repulsion (core_repulsion) in rho0, alpha and the Gaussians; zeros where there is none
  if constexpr (MODE == 0) {
    const double ra = g.r * kA0, w = pi[PAR_RHO0] + pj[PAR_RHO0];
    const double inv = rsq_nr(g.r * g.r + w * w);
    const double tt = ti * tj;
    const int Zi = (int)pi[PAR_Z], Zj = (int)pj[PAR_Z];
    double t2 = exp(-pi[PAR_ALPHA] * ra);
    if ((Zi == 7 || Zi == 8) && Zj == 1) t2 *= ra;
    const double t3 = exp(-pj[PAR_ALPHA] * ra);
    const double dg = -tt * (1.0 + t2 + t3) * kEV * (inv * inv * inv) * w;
    put(PV_REP, dg, dg);
    put(PV_ALPHA, -tt * kEV * inv * t2 * ra, -tt * kEV * inv * t3 * ra);
    const int ng = method == PYSEQM_AM1 ? 4 : (method == PYSEQM_PM3 ? 2 : 0);
    const double pre = tt / ra;
#pragma unroll 1
    for (int k = 0; k < 4; ++k) {
      double v[2][3];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const double* p = (s == 0 ? pi : pj) + PAR_GAUSS + 3 * k;
        const double dm = ra - p[2], e = k < ng ? pre * exp(-p[1] * dm * dm) : 0.0;
        v[s][0] = e;
        v[s][1] = -p[0] * dm * dm * e;
        v[s][2] = 2.0 * p[0] * p[1] * dm * e;
      }
#pragma unroll
      for (int x = 0; x < 3; ++x) put(PV_GAUSS + 3 * k + x, v[0][x], v[1][x]);
    }
  } else {
    put(PV_REP, 0.0, 0.0);
#pragma unroll
    for (int k = PV_ALPHA; k < kPV; ++k) put(k, 0.0, 0.0);
  }
}

// out[a][0][slot] += atom a's pair shares of dEelec/d(slot), out[a][1][slot] += the core repulsion's: the
// sums of its partial slots (fixed order), through its multipoles' Jacobian.  One wave per atom.
__global__ __launch_bounds__(256) void k_param_gather(pyseqm_layout_t L, int method, const double* __restrict__ part,
                                                      const double* __restrict__ jac, double* __restrict__ out) {
  const int a = blockIdx.x * 4 + threadIdx.x / 64;
  const int lane = threadIdx.x % 64;
  if (a >= L.natoms) return;  // uniform over the wave
  double acc[kPV];
#pragma unroll
  for (int k = 0; k < kPV; ++k) acc[k] = 0.0;
  for (int e = L.csr_off[a] + lane; e < L.csr_off[a + 1]; e += 64) {
    const double* src = part + (size_t)L.csr_idx[e] * kPV;
#pragma unroll
    for (int k = 0; k < kPV; ++k) acc[k] += src[k];
  }
#pragma unroll
  for (int k = 0; k < kPV; ++k) acc[k] = wave64(acc[k]);
  if (lane != 0) return;
  double* oe = out + (size_t)a * 48;
  double* on = oe + 24;
#pragma unroll
  for (int k = 0; k < kJacSlots; ++k) {
    const double* J = jac + ((size_t)a * kJacSlots + k) * 5;
    oe[kJacParam[k]] +=
        acc[PV_DD] * J[0] + acc[PV_QQ] * J[1] + acc[PV_R0] * J[2] + acc[PV_R1] * J[3] + acc[PV_R2] * J[4];
    on[kJacParam[k]] += acc[PV_REP] * J[2];
  }
  oe[PAR_ZS] += acc[PV_ZS];
  oe[PAR_ZP] += acc[PV_ZP];
  oe[PAR_BS] += acc[PV_BS];
  oe[PAR_BP] += acc[PV_BP];
  on[PAR_ALPHA] += acc[PV_ALPHA];
  const int ng = method == PYSEQM_AM1 ? 12 : (method == PYSEQM_PM3 ? 6 : 0);
#pragma unroll
  for (int k = 0; k < 12; ++k)
    if (k < ng) on[PAR_GAUSS + k] += acc[PV_GAUSS + k];
}

// The closed-form one-center part: E_A = sum_mu P_mumu U_mu + 1/2 sum P G1(P) over the atom's
// block (the one-center terms of the Fock build, fock.py:196-224), differentiated in U_ss, U_pp,
// g_ss, g_sp, g_pp, g_p2 and h_sp; with Y given, the same for sum Y (U + G1(P)) over the block.
// Writes every slot of out[a] (the pair passes add to it).
__global__ void k_param_onecenter(pyseqm_layout_t L, const double* __restrict__ P, const double* __restrict__ Y,
                                  double* __restrict__ out) {
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  if (a >= L.natoms) return;
  const int m = L.atom_mol[a];
  const int n = L.mol_norb[m];
  const double* Pm = P + L.mol_mat_off[m];
  const int ao = L.atom_ao[a];
  double* o = out + (size_t)a * 48;
  for (int k = 0; k < 48; ++k) o[k] = 0.0;
  const double pss = Pm[(size_t)ao * n + ao];
  if (!Y) {
    o[PAR_USS] = pss;
    o[PAR_GSS] = 0.25 * pss * pss;
    if (L.atom_Z[a] > 1) {
      double pd[10];
#pragma unroll
      for (int k = 0; k < 10; ++k) pd[k] = Pm[(size_t)(ao + kTriI[k]) * n + ao + kTriJ[k]];
      const double ppt = pd[2] + pd[5] + pd[9];
      const double psp2 = pd[1] * pd[1] + pd[3] * pd[3] + pd[6] * pd[6];
      const double ppd2 = pd[2] * pd[2] + pd[5] * pd[5] + pd[9] * pd[9];
      const double ppo2 = pd[4] * pd[4] + pd[7] * pd[7] + pd[8] * pd[8];
      o[PAR_UPP] = ppt;
      o[PAR_GSP] = pss * ppt - 0.5 * psp2;
      o[PAR_HSP] = -0.5 * pss * ppt + 1.5 * psp2;
      o[PAR_GPP] = 0.375 * ppd2 - 0.125 * ppt * ppt + 0.75 * ppo2;
      o[PAR_GP2] = 0.625 * (ppt * ppt - ppd2) - 1.25 * ppo2;
    }
    return;
  }
  // sum Y (U + G1(P)): diagonal elements once, off-diagonal pairs twice (both triangles)
  const double* Ym = Y + L.mol_mat_off[m];
  const double yss = Ym[(size_t)ao * n + ao];
  o[PAR_USS] = yss;
  o[PAR_GSS] = 0.5 * yss * pss;
  if (L.atom_Z[a] > 1) {
    double pd[10], yd[10];
#pragma unroll
    for (int k = 0; k < 10; ++k) {
      pd[k] = Pm[(size_t)(ao + kTriI[k]) * n + ao + kTriJ[k]];
      yd[k] = Ym[(size_t)(ao + kTriI[k]) * n + ao + kTriJ[k]];
    }
    const double ppt = pd[2] + pd[5] + pd[9], ypt = yd[2] + yd[5] + yd[9];
    const double ysp = yd[1] * pd[1] + yd[3] * pd[3] + yd[6] * pd[6];
    const double ypd = yd[2] * pd[2] + yd[5] * pd[5] + yd[9] * pd[9];
    const double ypo = yd[4] * pd[4] + yd[7] * pd[7] + yd[8] * pd[8];
    o[PAR_UPP] = ypt;
    o[PAR_GSP] = yss * ppt + ypt * pss - ysp;
    o[PAR_HSP] = -0.5 * (yss * ppt + ypt * pss) + 3.0 * ysp;
    o[PAR_GPP] = 0.75 * ypd - 0.25 * ypt * ppt + 1.5 * ypo;
    o[PAR_GP2] = 1.25 * (ypt * ppt - ypd) - 2.5 * ypo;
  }
}

// Diagonal core-Hamiltonian blocks: U on the diagonal plus the electron-core attractions
// collected from every tile the atom appears in (hcore.py:127-150), fixed summation order.
template <int G>
__global__ __launch_bounds__(256) void k_hcore_diag(pyseqm_layout_t L, const double* __restrict__ par,
                                                    const double* __restrict__ part, double* __restrict__ H) {
  const int a = blockIdx.x * (256 / G) + threadIdx.x / G;
  const int lane = threadIdx.x % G;
  if (a >= L.natoms) return;  // uniform over the lane group
  const double* p = par + (size_t)a * PYSEQM_NPAR;
  const int m = L.atom_mol[a];
  const int norb = L.mol_norb[m];
  double* Hm = H + L.mol_mat_off[m];
  const int ao = L.atom_ao[a];
  const int e0 = L.csr_off[a], e1 = L.csr_off[a + 1];
  if (L.atom_Z[a] > 1) {
    double acc[10];
    gather_slots_c<G>(part, L, e0, e1, lane, acc);
    acc[0] += p[PAR_USS];
    acc[2] += p[PAR_UPP];
    acc[5] += p[PAR_UPP];
    acc[9] += p[PAR_UPP];
    if (lane < 16) {
      const int mu = lane >> 2, nu = lane & 3;
      double v = acc[0];
#pragma unroll
      for (int k = 1; k < 10; ++k)
        if (k == tri_index(mu, nu)) v = acc[k];
      Hm[(size_t)(ao + mu) * norb + ao + nu] = v;
    }
  } else {
    double acc[1];
    gather_slots_c<G>(part, L, e0, e1, lane, acc);
    if (lane == 0) Hm[(size_t)ao * norb + ao] = acc[0] + p[PAR_USS];
  }
}

// Per-molecule sum of per-tile values (and optionally per-atom values): one block per molecule,
// threads stride over the molecule's tiles / atoms, fixed thread assignment, wave shuffle trees and
// a fixed-order sum of the wave totals.
template <int NT>
__global__ __launch_bounds__(NT) void k_mol_sum(pyseqm_layout_t L, const double* __restrict__ tile_v,
                                                const double* __restrict__ atom_v,
                                                const unsigned char* __restrict__ active, double* __restrict__ out) {
  __shared__ double wsum[NT / 64];
  const int m = blockIdx.x;
  if (active && !active[m]) return;
  const int tid = threadIdx.x;
  // eight independent partial sums per thread keep eight loads in flight (a single running sum
  // waits out one memory round trip per element); combined in a fixed order
  double acc[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  auto add_range = [&](const double* v, int b, int e) {
    int t = b + tid;
    for (; t + 7 * NT < e; t += 8 * NT) {
#pragma unroll
      for (int u = 0; u < 8; ++u) acc[u] += v[t + u * NT];
    }
    for (; t < e; t += NT) acc[0] += v[t];
  };
  for (int kind = 0; kind < 3; ++kind) {
    const int* off = L.mol_tile_off + kind * (L.nmol + 1);
    add_range(tile_v, off[m], off[m + 1]);
  }
  if (atom_v) add_range(atom_v, L.mol_atom_off[m], L.mol_atom_off[m + 1]);
  double s = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
  s = wave_sum(s);
  if ((tid & 63) == 0) wsum[tid >> 6] = s;
  __syncthreads();
  if (tid == 0) {
    double r = 0.0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) r += wsum[w];
    out[m] = r;
  }
}

}  // namespace

namespace pyseqm {
void launch_mol_sum(const pyseqm_layout_t* L, const double* tile_v, const double* atom_v,
                    const unsigned char* active, double* out, hipStream_t s) {
  if (L->nmol <= 0) return;
  const long long nt = (long long)L->ntile[0] + L->ntile[1] + L->ntile[2];
  if (nt > 2048LL * L->nmol)
    k_mol_sum<1024><<<L->nmol, 1024, 0, s>>>(*L, tile_v, atom_v, active, out);
  else
    k_mol_sum<64><<<L->nmol, 64, 0, s>>>(*L, tile_v, atom_v, active, out);
}
}  // namespace pyseqm

namespace {
// Core-core repulsion of an explicit pair list (energy.py:91-134): one thread per pair, gam given.
__global__ void k_core_repulsion_pairs(long long npairs, int method, const int* __restrict__ idxi,
                                       const int* __restrict__ idxj, const double* __restrict__ rij,
                                       const double* __restrict__ gam, const double* __restrict__ par,
                                       double* __restrict__ out) {
  const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= npairs) return;
  const double* pi = par + (size_t)idxi[k] * PYSEQM_NPAR;
  const double* pj = par + (size_t)idxj[k] * PYSEQM_NPAR;
  out[k] = core_repulsion(method, (int)pi[PAR_Z], (int)pj[PAR_Z], rij[k], gam[k], pi, pj);
}
}  // namespace

extern "C" int pyseqm_core_repulsion_pairs(long long npairs, int method, const int* idxi, const int* idxj,
                                           const double* rij, const double* gam, const double* atom_par,
                                           double* enuc_pair, void* stream) {
  if (npairs < 0 || method < PYSEQM_MNDO || method > PYSEQM_PM3) return PYSEQM_EINVAL;
  if (npairs == 0) return PYSEQM_OK;
  k_core_repulsion_pairs<<<(unsigned)((npairs + 255) / 256), 256, 0, (hipStream_t)stream>>>(
      npairs, method, idxi, idxj, rij, gam, atom_par, enuc_pair);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}

namespace {
template <bool XL>
int launch_pair_forces(const pyseqm_layout_t* L, int method, const double* coords, const double* atom_par,
                       const double* P, const double* D, double h, double* part, double* forces, void* stream) {
  if (!L || method < PYSEQM_MNDO || method > PYSEQM_PM3 || !(h > 0.0)) return PYSEQM_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  const int n0 = L->ntile[0], n1 = L->ntile[1], n2 = L->ntile[2];
  if (merge_kinds(L)) {
    if (n0 + n1 + n2)
      k_pair_forces<ALL, XL><<<n0 + n1 + n2, 64, 0, s>>>(*L, method, 0, coords, atom_par, P, D, part);
  } else {
    if (n0) k_pair_forces<XX, XL><<<n0, 64, 0, s>>>(*L, method, 0, coords, atom_par, P, D, part);
    if (n1) k_pair_forces<XH, XL><<<n1, 64, 0, s>>>(*L, method, n0, coords, atom_par, P, D, part);
    if (n2) k_pair_forces<HH, XL><<<n2, 64, 0, s>>>(*L, method, n0 + n1, coords, atom_par, P, D, part);
  }
  if (L->natoms) {
    if (lanes_per_atom(L) == 64)
      k_atom_forces<64><<<(L->natoms + 3) / 4, 256, 0, s>>>(*L, part, forces);
    else
      k_atom_forces<16><<<(L->natoms + 15) / 16, 256, 0, s>>>(*L, part, forces);
  }
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}
}  // namespace

extern "C" int pyseqm_pair_forces(const pyseqm_layout_t* L, int method, const double* coords,
                                  const double* atom_par, const double* P, double h, double* part, double* forces,
                                  void* stream) {
  return launch_pair_forces<false>(L, method, coords, atom_par, P, nullptr, h, part, forces, stream);
}

extern "C" int pyseqm_pair_forces_xl(const pyseqm_layout_t* L, int method, const double* coords,
                                     const double* atom_par, const double* D, const double* P, double h,
                                     double* part, double* forces, void* stream) {
  if (!D || !P) return PYSEQM_EINVAL;
  return launch_pair_forces<true>(L, method, coords, atom_par, P, D, h, part, forces, stream);
}

extern "C" long long pyseqm_param_grad_workspace(const pyseqm_layout_t* L) {
  if (!L || L->natoms < 0) return -1;
  const long long nt = (long long)L->ntile[0] + L->ntile[1] + L->ntile[2];
  return nt * 16 * kPV + (long long)L->natoms * kJacSlots * 5;
}

namespace {
// ws: the tiles' 23-wide partials, then the atoms' Jacobians (pyseqm_param_grad_workspace)
template <int MODE>
int launch_param_grad(const pyseqm_layout_t* L, int method, const double* coords, const double* atom_par,
                      const double* P, const double* Y, double hrel, double* ws, double* out, void* stream) {
  if (!L || method < PYSEQM_MNDO || method > PYSEQM_PM3 || !(hrel > 0.0)) return PYSEQM_EINVAL;
  if (L->natoms == 0) return PYSEQM_OK;
  hipStream_t s = (hipStream_t)stream;
  const size_t nt = (size_t)L->ntile[0] + L->ntile[1] + L->ntile[2];
  double* part = ws;
  double* jac = ws + nt * 16 * kPV;
  k_param_onecenter<<<(L->natoms + 127) / 128, 128, 0, s>>>(*L, P, Y, out);
  k_param_jacobian<<<(L->natoms * kJacSlots + 127) / 128, 128, 0, s>>>(*L, atom_par, hrel, jac);
  int base = 0;
  if (L->ntile[0])
    k_pair_param_grad<XX, MODE><<<L->ntile[0], 64, 0, s>>>(*L, method, base, coords, atom_par, P, Y, part);
  base += L->ntile[0];
  if (L->ntile[1])
    k_pair_param_grad<XH, MODE><<<L->ntile[1], 64, 0, s>>>(*L, method, base, coords, atom_par, P, Y, part);
  base += L->ntile[1];
  if (L->ntile[2])
    k_pair_param_grad<HH, MODE><<<L->ntile[2], 64, 0, s>>>(*L, method, base, coords, atom_par, P, Y, part);
  k_param_gather<<<(L->natoms + 3) / 4, 256, 0, s>>>(*L, method, part, jac, out);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}
}  // namespace

extern "C" int pyseqm_param_grad(const pyseqm_layout_t* L, int method, const double* coords, const double* atom_par,
                                 const double* P, double hrel, double* rec, double* part, double* out,
                                 void* stream) {
  (void)part;
  return launch_param_grad<0>(L, method, coords, atom_par, P, nullptr, hrel, rec, out, stream);
}

extern "C" int pyseqm_fock_param_vjp(const pyseqm_layout_t* L, int method, const double* coords,
                                     const double* atom_par, const double* P, const double* Y, double hrel,
                                     double* rec, double* part, double* out, void* stream) {
  if (!Y) return PYSEQM_EINVAL;
  (void)part;
  return launch_param_grad<2>(L, method, coords, atom_par, P, Y, hrel, rec, out, stream);
}

extern "C" int pyseqm_atom_setup(const pyseqm_layout_t* L, double* atom_par, void* stream) {
  if (!L || L->natoms < 0) return PYSEQM_EINVAL;
  if (L->natoms == 0) return PYSEQM_OK;
  hipStream_t s = (hipStream_t)stream;
  k_atom_setup<<<(L->natoms + 127) / 128, 128, 0, s>>>(*L, atom_par);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}

extern "C" int pyseqm_pair_integrals(const pyseqm_layout_t* L, int method, const double* coords,
                                     const double* atom_par, double* w_xx, double* w_xh, double* w_hh,
                                     double* H, double* part, double* enuc_tile, double* enuc_mol,
                                     double* enuc_pair, const int* pair_ref, void* stream) {
  if (!L || method < PYSEQM_MNDO || method > PYSEQM_PM3) return PYSEQM_EINVAL;
  if (enuc_pair && !pair_ref) return PYSEQM_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  const int n0 = L->ntile[0], n1 = L->ntile[1], n2 = L->ntile[2];
  auto launch = [&](auto kind, int count, int base) {
    if (count)
      k_pair_tiles<decltype(kind)::value><<<count, 64, 0, s>>>(*L, method, base, coords, atom_par, w_xx, w_xh, w_hh, H,
                                                               part, enuc_tile, enuc_pair, pair_ref);
  };
  if (merge_kinds(L)) {
    launch(std::integral_constant<int, ALL>(), n0 + n1 + n2, 0);
  } else {
    launch(std::integral_constant<int, XX>(), n0, 0);
    launch(std::integral_constant<int, XH>(), n1, n0);
    launch(std::integral_constant<int, HH>(), n2, n0 + n1);
  }
  if (L->natoms) {
    if (lanes_per_atom(L) == 64)
      k_hcore_diag<64><<<(L->natoms + 3) / 4, 256, 0, s>>>(*L, atom_par, part, H);
    else
      k_hcore_diag<16><<<(L->natoms + 15) / 16, 256, 0, s>>>(*L, atom_par, part, H);
  }
  pyseqm::launch_mol_sum(L, enuc_tile, nullptr, nullptr, enuc_mol, s);
  return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH;
}
