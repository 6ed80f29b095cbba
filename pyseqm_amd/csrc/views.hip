// The packed batch in the reference's layouts: padded matrices (nmol, 4 molsize, 4 molsize), the
// block array of the core Hamiltonian (hcore.py:155-179), dense two-center integrals (npairs, 10, 10)
// and per-orbital atomic charges (scf_loop.py:2376-2387).  Every index follows from the molecule's
// atom counts, so no index arrays are built or read, and every output element is written (zeros
// included): each kernel moves its input and its output once.  What bounds them is HBM; the index
// lists they stand in for took the host 25 ms per batch of 128 alkanes of 2-30 carbons.
#include "common.h"

using namespace pyseqm;

namespace {

// orbital of padded row p (component p % 4 of atom p / 4) in a molecule of nat atoms, nh of them heavy,
// or -1: hydrogens carry one orbital, the last atoms of a row are padding
__device__ inline int orbital_of(int p, int nat, int nh) {
  const int a = p >> 2;
  if (a < nh) return p;
  return (a < nat && (p & 3) == 0) ? 4 * nh + a - nh : -1;
}
__device__ inline void counts_of(const pyseqm_layout_t& L, int m, int& nat, int& nh, int& n) {
  nat = L.mol_atom_off[m + 1] - L.mol_atom_off[m];
  n = L.mol_norb[m];
  nh = (n - nat) / 3;  // n = 4 nh + (nat - nh)
}

constexpr int kViewRows = 8;  // padded rows per block

// MODE 0: every element; 1: the upper triangle of the padded matrix, zero below; 2: that triangle as
// 4 x 4 blocks (atom i, atom j)
template <int MODE>
__global__ __launch_bounds__(256) void k_to_padded(pyseqm_layout_t L, int molsize, const double* __restrict__ X,
                                                   double* __restrict__ out) {
  const int m = blockIdx.x, w = 4 * molsize;
  int nat, nh, n;
  counts_of(L, m, nat, nh, n);
  const double* x = X + L.mol_mat_off[m];
  double* o = out + (size_t)m * w * w;
  const int r1 = min(w, (int)(blockIdx.y + 1) * kViewRows);
  for (int r = blockIdx.y * kViewRows; r < r1; ++r) {
    const int ro = orbital_of(r, nat, nh);
    for (int c = threadIdx.x; c < w; c += 256) {
      const int co = orbital_of(c, nat, nh);
      double v = 0.0;
      if (ro >= 0 && co >= 0 && (MODE == 0 || r <= c)) v = x[(size_t)ro * n + co];
      if (MODE == 2)
        o[((size_t)(r >> 2) * molsize + (c >> 2)) * 16 + (r & 3) * 4 + (c & 3)] = v;
      else
        o[(size_t)r * w + c] = v;
    }
  }
}

__global__ __launch_bounds__(256) void k_from_padded(pyseqm_layout_t L, int molsize, const double* __restrict__ Xp,
                                                     double* __restrict__ out) {
  const int m = blockIdx.x, w = 4 * molsize;
  int nat, nh, n;
  counts_of(L, m, nat, nh, n);
  const double* x = Xp + (size_t)m * w * w;
  double* o = out + L.mol_mat_off[m];
  const int r1 = min(n, (int)(blockIdx.y + 1) * kViewRows);
  for (int r = blockIdx.y * kViewRows; r < r1; ++r) {
    const int rp = r < 4 * nh ? r : 4 * (r - 3 * nh);
    for (int c = threadIdx.x; c < n; c += 256)
      o[(size_t)r * n + c] = x[(size_t)rp * w + (c < 4 * nh ? c : 4 * (c - 3 * nh))];
  }
}

// index of pair (i, j), i < j local, in the reference's order within a molecule of nat atoms
__device__ inline long long pair_index(int i, int j, int nat) {
  return (long long)i * nat - (long long)i * (i + 1) / 2 + (j - i - 1);
}

__global__ __launch_bounds__(64) void k_pair_ref(pyseqm_layout_t L, const long long* __restrict__ pair_base,
                                                 int* __restrict__ out) {
  const Tile t = load_tile(L.tiles, blockIdx.x);
  int i, j;
  const bool ok = lane_pair(t, threadIdx.x, i, j);
  const int a0 = L.mol_atom_off[t.mol], nat = L.mol_atom_off[t.mol + 1] - a0;
  out[(size_t)blockIdx.x * 64 + threadIdx.x] = ok ? (int)(pair_base[t.mol] + pair_index(i - a0, j - a0, nat)) : -1;
}

// One tile by a workgroup: its integrals (rows of packed lanes) are read in order into LDS and written a pair's 100
// values at a time, two per thread; heavy-H pairs fill column 0, H-H pairs element 0 (the rest is zero).
// The LDS row stride is odd, so a pair's values lie on distinct banks.
constexpr int kRefThreads = 1024;
template <int KIND>
__device__ __forceinline__ void w_reference_tile(const pyseqm_layout_t& L, int tile,
                                                 const long long* __restrict__ pair_base,
                                                 const double* __restrict__ w, double* __restrict__ out, double* buf,
                                                 long long* ref) {
  constexpr int NW = KIND == 0 ? 100 : (KIND == 1 ? 10 : 1);
  const Tile t = load_tile(L.tiles, tile);
  const int S = tile_wstride(t), nv = t.diag ? t.nrow * (t.nrow - 1) / 2 : t.nrow * t.ncol;
  if (threadIdx.x < 64) {
    int i, j;
    if (lane_pair(t, threadIdx.x, i, j)) {
      const int a0 = L.mol_atom_off[t.mol], nat = L.mol_atom_off[t.mol + 1] - a0;
      ref[lane_rank(t, threadIdx.x)] = pair_base[t.mol] + pair_index(i - a0, j - a0, nat);
    }
  }
  const double* src = w + L.tile_woff[tile];
#pragma unroll 4
  for (int e = threadIdx.x; e < NW * S; e += kRefThreads) {
    const int q = e / S, p = e - q * S;
    const double v = src[e];
    if (p < nv) buf[q * 65 + p] = v;
  }
  __syncthreads();
#pragma unroll 2
  for (int e = threadIdx.x; e < nv * 50; e += kRefThreads) {
    const int p = e / 50, q = 2 * (e - p * 50);
    double2 v = make_double2(0.0, 0.0);
    if (KIND == 0)
      v = make_double2(buf[q * 65 + p], buf[(q + 1) * 65 + p]);
    else if (KIND == 1)
      v.x = q % 10 == 0 ? buf[(q / 10) * 65 + p] : 0.0;
    else
      v.x = q == 0 ? buf[p] : 0.0;
    *reinterpret_cast<double2*>(out + ref[p] * 100 + q) = v;
  }
}

// All tiles in one launch, heavy-heavy ones first (a launch per kind with 256 threads, whose loops wait for
// memory ~25 times: 16 clusters of 24 waters 28 us, 10 here; 128 alkanes of 2-30 carbons 57, 53).
__global__ __launch_bounds__(kRefThreads) void k_w_reference(pyseqm_layout_t L,
                                                             const long long* __restrict__ pair_base,
                                                             const double* __restrict__ w_xx,
                                                             const double* __restrict__ w_xh,
                                                             const double* __restrict__ w_hh,
                                                             double* __restrict__ out) {
  __shared__ double buf[100 * 65];
  __shared__ long long ref[64];
  const int b = blockIdx.x, n0 = L.ntile[0], n1 = n0 + L.ntile[1];
  if (b < n0)
    w_reference_tile<0>(L, b, pair_base, w_xx, out, buf, ref);
  else if (b < n1)
    w_reference_tile<1>(L, b, pair_base, w_xh, out, buf, ref);
  else
    w_reference_tile<2>(L, b, pair_base, w_hh, out, buf, ref);
}

// The reference's atom and pair lists (Parser, basics.py:199-403) of a padded batch in which every pair of real atoms
// counts: one block per padded atom (m, i), threads over the partners j > i.  Rows are sorted (padding last),
// so atom i of molecule m is number atom_off[m] + i and its pairs are in row-major order.  As index arithmetic
// on whole padded tensors this took some 35 launches, 10 to 15 us of host time each.  beyond: counts the pairs
// that are not closer than `cutoff` (NaN included); the caller drops them.
__global__ __launch_bounds__(64) void k_pair_lists(int molsize, const long long* __restrict__ species,
                                                   const double* __restrict__ xyz,
                                                   const long long* __restrict__ atom_off,
                                                   const long long* __restrict__ pair_off, double cutoff,
                                                   long long* __restrict__ atoms, long long natoms,
                                                   long long* __restrict__ pairs, long long npairs,
                                                   double* __restrict__ xij, double* __restrict__ rij,
                                                   int* __restrict__ beyond) {
  const long long m = blockIdx.y, i = blockIdx.x;
  const long long a0 = atom_off[m], nat = atom_off[m + 1] - a0;
  if (i >= nat) return;
  const long long* z = species + m * molsize;
  const double* x = xyz + m * molsize * 3;
  const long long zi = z[i], w = molsize;
  if (threadIdx.x == 0) {  // Z, maskd, atom_molid
    atoms[a0 + i] = zi;
    atoms[natoms + a0 + i] = m * w * w + i * (w + 1);
    atoms[2 * natoms + a0 + i] = m;
  }
  const long long p0 = pair_off[m] + pair_index((int)i, (int)i + 1, (int)nat);
  for (long long j = i + 1 + threadIdx.x; j < nat; j += 64) {
#pragma clang fp contract(off)
    const long long p = p0 + (j - i - 1);
    const long long v[7] = {m, zi, z[j], a0 + i, a0 + j, m * w * w + i * w + j, m * w * w + j * w + i};
#pragma unroll
    for (int q = 0; q < 7; ++q) pairs[q * npairs + p] = v[q];  // molecule, ni, nj, idxi, idxj, mask, mask_l
    const double d0 = x[3 * j] - x[3 * i], d1 = x[3 * j + 1] - x[3 * i + 1], d2 = x[3 * j + 2] - x[3 * i + 2];
    const double r = sqrt(d0 * d0 + d1 * d1 + d2 * d2);
    rij[p] = r;
    xij[3 * p] = d0 / r;
    xij[3 * p + 1] = d1 / r;
    xij[3 * p + 2] = d2 / r;
    if (!(r < cutoff)) atomicAdd(beyond, 1);
  }
}

// charge[i][a] of the reference's per-orbital charges: with v row i of V squared, heavy atom a takes
// v[a], v[nh + a], v[2 nh + a], v[3 nh + a] (the reference's reshape), hydrogen a takes its orbital
__global__ __launch_bounds__(256) void k_orbital_charges(pyseqm_layout_t L, int molsize, const double* __restrict__ V,
                                                         long long sm, long long sr, long long sc,
                                                         double* __restrict__ out) {
  const int m = blockIdx.x, w = 4 * molsize;
  int nat, nh, n;
  counts_of(L, m, nat, nh, n);
  const double* v = V + m * sm;
  double* o = out + (size_t)m * w * molsize;
  const int i1 = min(w, (int)(blockIdx.y + 1) * kViewRows);
  for (int i = blockIdx.y * kViewRows; i < i1; ++i)
    for (int a = threadIdx.x; a < molsize; a += 256) {
      double q = 0.0;
      if (i < n && a < nh) {
        for (int c = 0; c < 4; ++c) {
          const double x = v[i * sr + (long long)(c * nh + a) * sc];
          q += x * x;
        }
      } else if (i < n && a < nat) {
        const double x = v[i * sr + (long long)(3 * nh + a) * sc];
        q = x * x;
      }
      o[(size_t)i * molsize + a] = q;
    }
}

// Packed eigenpairs (column j of Q: vector j, lam[orb_off[m] + j]) as zero-padded eigenvalues e[m][w] and
// vectors V[m][nmax][nmax], the identity beyond the block: the basis vectors of padding rows, as a padded
// solve would return them.
__global__ __launch_bounds__(256) void k_evec_view(pyseqm_layout_t L, int w, int nmax,
                                                   const long long* __restrict__ orb_off,
                                                   const double* __restrict__ lam, const double* __restrict__ Q,
                                                   double* __restrict__ e, double* __restrict__ V,
                                                   int* __restrict__ fail) {
  const int m = blockIdx.x, n = L.mol_norb[m];
  const double* q = Q + L.mol_mat_off[m];
  double* v = V + (size_t)m * nmax * nmax;
  const int r1 = min(nmax, (int)(blockIdx.y + 1) * kViewRows);
  for (int r = blockIdx.y * kViewRows; r < r1; ++r)
    for (int c = threadIdx.x; c < nmax; c += 256)
      v[(size_t)r * nmax + c] = (r < n && c < n) ? q[(size_t)r * n + c] : (r == c ? 1.0 : 0.0);
  if (blockIdx.y == 0)
    for (int c = threadIdx.x; c < w; c += 256) {
      const double x = c < n ? lam[orb_off[m] + c] : 0.0;
      e[(size_t)m * w + c] = x;
      if (!(fabs(x) < INFINITY)) atomicAdd(fail, 1);
    }
}

dim3 view_grid(const pyseqm_layout_t& L, int molsize) {
  return dim3(L.nmol, (4 * molsize + kViewRows - 1) / kViewRows);
}
int launched() { return hipGetLastError() == hipSuccess ? PYSEQM_OK : PYSEQM_ELAUNCH; }

}  // namespace

extern "C" int pyseqm_to_padded(const pyseqm_layout_t* L, int molsize, int mode, const double* X, double* out,
                                void* stream) {
  if (!L || molsize < 1 || mode < 0 || mode > 2) return PYSEQM_EINVAL;
  if (L->nmol == 0) return PYSEQM_OK;
  const dim3 g = view_grid(*L, molsize);
  hipStream_t s = (hipStream_t)stream;
  if (mode == 0)
    k_to_padded<0><<<g, 256, 0, s>>>(*L, molsize, X, out);
  else if (mode == 1)
    k_to_padded<1><<<g, 256, 0, s>>>(*L, molsize, X, out);
  else
    k_to_padded<2><<<g, 256, 0, s>>>(*L, molsize, X, out);
  return launched();
}

extern "C" int pyseqm_from_padded(const pyseqm_layout_t* L, int molsize, const double* Xp, double* out, void* stream) {
  if (!L || molsize < 1) return PYSEQM_EINVAL;
  if (L->nmol == 0) return PYSEQM_OK;
  k_from_padded<<<view_grid(*L, molsize), 256, 0, (hipStream_t)stream>>>(*L, molsize, Xp,
                                                                                                         out);
  return launched();
}

extern "C" int pyseqm_pair_ref(const pyseqm_layout_t* L, const long long* pair_base, int* out, void* stream) {
  if (!L) return PYSEQM_EINVAL;
  const int nt = L->ntile[0] + L->ntile[1] + L->ntile[2];
  if (nt == 0) return PYSEQM_OK;
  k_pair_ref<<<nt, 64, 0, (hipStream_t)stream>>>(*L, pair_base, out);
  return launched();
}

extern "C" int pyseqm_w_reference(const pyseqm_layout_t* L, const long long* pair_base, const double* w_xx,
                                  const double* w_xh, const double* w_hh, double* out, void* stream) {
  if (!L) return PYSEQM_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  const int tiles = L->ntile[0] + L->ntile[1] + L->ntile[2];
  if (tiles) k_w_reference<<<tiles, kRefThreads, 0, s>>>(*L, pair_base, w_xx, w_xh, w_hh, out);
  return launched();
}

extern "C" int pyseqm_pair_lists(int nmol, int molsize, const long long* species, const double* xyz,
                                 const long long* atom_off, const long long* pair_off, double cutoff,
                                 long long* atoms, long long natoms, long long* pairs, long long npairs, double* xij,
                                 double* rij, int* beyond, void* stream) {
  if (nmol < 0 || nmol > 65535 || molsize < 1 || natoms < 0 || npairs < 0 || !beyond) return PYSEQM_EINVAL;
  if (nmol == 0 || natoms == 0) return PYSEQM_OK;
  k_pair_lists<<<dim3(molsize, nmol), 64, 0, (hipStream_t)stream>>>(molsize, species, xyz, atom_off, pair_off, cutoff,
                                                                    atoms, natoms, pairs, npairs, xij, rij, beyond);
  return launched();
}

extern "C" int pyseqm_evec_view(const pyseqm_layout_t* L, int molsize, int nmax, const long long* orb_off,
                                const double* lam, const double* Q, double* e, double* V, int* fail, void* stream) {
  if (!L || molsize < 1 || nmax < 1 || !orb_off || !fail || nmax > 4 * molsize) return PYSEQM_EINVAL;
  if (L->nmol == 0) return PYSEQM_OK;
  const dim3 g(L->nmol, (nmax + kViewRows - 1) / kViewRows);
  k_evec_view<<<g, 256, 0, (hipStream_t)stream>>>(*L, 4 * molsize, nmax, orb_off, lam, Q, e, V, fail);
  return launched();
}

extern "C" int pyseqm_orbital_charges(const pyseqm_layout_t* L, int molsize, const double* V, long long stride_mol,
                                      long long stride_row, long long stride_col, double* out, void* stream) {
  if (!L || molsize < 1) return PYSEQM_EINVAL;
  if (L->nmol == 0) return PYSEQM_OK;
  k_orbital_charges<<<view_grid(*L, molsize), 256, 0, (hipStream_t)stream>>>(
      *L, molsize, V, stride_mol, stride_row, stride_col, out);
  return launched();
}
