// Batched SCF: thousands of small molecules of uneven size.  The control logic
// of iter (src/SCF/iter.F90:340-1041: level shift, convergence test, recompute
// with shift 0, ready/iredy) runs on the device for every molecule.
//
// A molecule of up to 64 orbitals is one workgroup's from start to end
// (k_bscf_lds): Fock build, energy, control, eigensolve and density in its
// LDS, cnvg.  Larger ones iterate together, a launch per phase over all of
// them: control (shift, mode) -> fock2 (batched) -> helect -> control
// (energy, test) -> block-Jacobi eigensolve + density (k_batch_eig.hip) -> cnvg
// (batched) -> control (PL, frontier levels, newdg) -> Pa = P / 2.  Molecules
// that have converged drop out by a flag.
#include <algorithm>
#include <chrono>
#include <climits>
#include <cmath>
#include <type_traits>
#include <vector>

#include "common.h"
#include "k_batch.h"
#include "k_fock.h"
#include "k_fock_body.h"
#include "k_jacobi_step.h"

namespace mhip {
namespace {

__device__ __forceinline__ double beig_flops(int n, int nocc, long long nrot, bool warm) {
  const double dn = n, tn = 0.5 * dn * (dn + 1.0);
  return 12.0 * dn * (double)nrot + (warm ? 2.0 * dn * dn * dn + 2.0 * dn * tn : 0.0) + 2.0 * tn * nocc;
}

constexpr double kEnrgy = 23.060547830619029;  // fpc_9, eV -> kcal/mol

// ---- control, part 1: shift and Fock mode (iter.F90:340-420) ---------------
__device__ void ctl_pre(BatchState& s) {
  if (s.recompute) {
    // label 320 again: F from H with the shift set to zero, same iteration
    s.mode = kInitH;
  } else {
    s.niter += 1;
    const double bshift = -80.0;
    s.mode = kInitH;
    if (fabs(s.shift) > 1e-10) {
      if (s.niter > 1) {
        if (s.newdg) {
          if (s.diff > 0.0) {
            s.shift = 1.0;
            if (s.diff > 1) s.newdg = 0;
          } else {
            s.shift = -0.1;
          }
        } else {
          s.shift = s.ten + s.eig_lumo - s.eig_homo + s.shift;
        }
        if (s.diff > 0.0) {
          if (s.shift > 4.0) s.shfmax = 4.5;
          if (s.shift > s.shfmax) s.shfmax = fmax(s.shfmax - 0.5, 0.0);
        }
        s.shift = fmax(-20.0, fmin(s.shfmax, s.shift));
        if (fabs(s.shift - s.shfmax) < 1e-5) s.shfmax += 0.01;
        (void)bshift;
      }
      if (s.pl > 0.005) {
        s.shftbo = s.shiftb;
        s.shfto = s.shift;
      } else {
        s.shiftb = s.shftbo;
        s.shift = s.shfto;
      }
      s.mode = kInitShift;
    }
  }
}

__global__ void k_bctl_pre(int nmol, const int* __restrict__ list, BatchState* __restrict__ st, int* __restrict__ act,
                           int* __restrict__ mode, int* __restrict__ niter_out,
                           double* __restrict__ shift_out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nmol) return;
  const int m = list[i];
  BatchState s = st[m];
  act[m] = !s.done;
  if (s.done) return;
  ctl_pre(s);
  mode[m] = s.mode;
  niter_out[m] = s.niter;
  shift_out[m] = s.shift;
  st[m] = s;
}

// ---- control, part 2: energy and convergence test (iter.F90:640-700) -------
// Sets done, recompute (F again, with the shift at zero) or do_eig.
__device__ void ctl_mid(BatchState& s, double ee) {
  s.do_eig = 0;
  s.ee = ee;
  if (!isfinite(s.ee)) {
    s.done = 1;
    s.converged = 0;
    return;
  }
  s.escf = (s.ee + s.enuclr) * kEnrgy + s.atheat;
  if (s.niter >= s.itrmax) {
    s.done = 1;
    return;
  }
  s.recompute = 0;
  s.diff = s.escf - s.eold;
  if (s.diff > 0) s.ten = s.ten - 1.0;
  else s.ten = s.ten * 0.975 + 0.05;
  s.sellim = fmax(s.selcon, 1e-15 * fmax(fabs(s.ee), 1.0));
  if (s.niter > 4 && (s.pl == 0.0 || (s.pl < s.pltest && fabs(s.diff) < s.sellim)) && s.ready) {
    if (fabs(s.shift) < 1e-10) {
      s.converged = 1;
      s.done = 1;
      return;
    }
    s.shift = 0.0;
    s.shiftb = 0.0;
    s.recompute = 1;
    return;
  }
  s.ready = s.iredy > 0 && (fabs(s.diff) < s.sellim * 10.0 || s.pl == 0.0);
  s.iredy += 1;
  s.eold = s.escf;
  s.do_eig = 1;
}

__global__ void k_bctl_mid(int nmol, const int* __restrict__ list, BatchState* __restrict__ st, const double* __restrict__ ee,
                           int* __restrict__ do_eig) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nmol) return;
  const int m = list[i];
  BatchState s = st[m];
  do_eig[m] = 0;
  if (s.done) return;
  ctl_mid(s, ee[m]);
  do_eig[m] = s.do_eig;
  st[m] = s;
}

// ---- eigensolve + density, one workgroup per molecule ------------------------
__device__ __forceinline__ int rr_index(int idx, int r, int np) {
  return idx == 0 ? 0 : 1 + ((r + idx - 1) % (np - 1));
}

template <int NT>
__device__ double wg_max(double v, double* red) {
  red[threadIdx.x] = v;
  __syncthreads();
  for (int w = NT / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
    __syncthreads();
  }
  const double r = red[0];
  __syncthreads();
  return r;
}

// what one eigensolve did
struct EigCount {
  int nrot, sweeps;
};

__device__ __forceinline__ void eig_done(const BatchMol& M, BatchState& s, EigCount c, bool warm) {
  if (threadIdx.x != 0) return;
  s.eig_rot += c.nrot;
  s.eig_flops += beig_flops(M.n, M.nocc, c.nrot, warm);
  s.sweeps += c.sweeps;
  s.last_sweeps = c.sweeps;
  s.stuck |= c.sweeps >= s.max_sweeps;
  s.ndiag += 1;
  s.have_c = 1;
}

// Eigenvectors of M.f (warm: from M.C) into M.C, ascending, the levels into
// M.eig, and, with nocc > 0, the packed density into M.p.  Matrices in global
// memory.
template <int NT>
__device__ EigCount beig_global(const BatchMol& M, double* f, bool warm, double tol, int max_sweeps, bool density) {
  const int n = M.n, tid = threadIdx.x;
  __shared__ double red[NT];
  __shared__ double cs[kMaxBatchN / 2], sn[kMaxBatchN / 2];
  __shared__ int pp[kMaxBatchN / 2], qq[kMaxBatchN / 2];
  __shared__ int rank[kMaxBatchN];
  __shared__ int nrot;
  __syncthreads();
  if (tid == 0) nrot = 0;
  int sweeps = 0;
  double* A = M.A;
  double* C = M.C;
  double* T = M.T;
  // eigenvectors_LAPACK: F(i,i) += i * 1e-10, in place
  for (int i = tid; i < n; i += NT) f[(long long)i * (i + 1) / 2 + i] += (double)(i + 1) * 1.0e-10;
  __syncthreads();
  auto F = [&](int r, int c) -> double {
    return r >= c ? f[(long long)r * (r + 1) / 2 + c] : f[(long long)c * (c + 1) / 2 + r];
  };
  if (warm) {
    // T = F C, A = C^T T
    for (int e = tid; e < n * n; e += NT) {
      const int r = e % n, c = e / n;
      double s = 0.0;
      for (int k = 0; k < n; ++k) s += F(r, k) * C[k + c * n];
      T[e] = s;
    }
    __syncthreads();
    for (int e = tid; e < n * n; e += NT) {
      const int r = e % n, c = e / n;
      double s = 0.0;
      for (int k = 0; k < n; ++k) s += C[k + r * n] * T[k + c * n];
      A[e] = s;
    }
  } else {
    for (int e = tid; e < n * n; e += NT) {
      const int r = e % n, c = e / n;
      A[e] = F(r, c);
      C[e] = (r == c) ? 1.0 : 0.0;
    }
  }
  __syncthreads();
  const int np = (n + 1) & ~1;
  const int npair = np / 2;
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    double off = 0.0, dg = 0.0;
    for (int e = tid; e < n * n; e += NT) {
      const int r = e % n, c = e / n;
      if (r == c) dg = fmax(dg, fabs(A[e]));
      else off = fmax(off, fabs(A[e]));
    }
    off = wg_max<NT>(off, red);
    dg = wg_max<NT>(dg, red);
    if (off <= tol * fmax(dg, 1.0)) break;
    ++sweeps;
    for (int r = 0; r < np - 1; ++r) {
      for (int k = tid; k < npair; k += NT) {
        int p = rr_index(k, r, np), q = rr_index(np - 1 - k, r, np);
        if (p > q) { const int t = p; p = q; q = t; }
        double c = 1.0, s = 0.0;
        if (q < n) {
          const double app = A[p + p * n], aqq = A[q + q * n], apq = A[p + q * n];
          if (fabs(apq) > 1.0e-300 && fabs(apq) > 1.0e-18 * sqrt(fabs(app * aqq))) {
            const double theta = (aqq - app) / (2.0 * apq);
            const double t = (theta >= 0.0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
            c = 1.0 / sqrt(t * t + 1.0);
            s = t * c;
            atomicAdd(&nrot, 1);
          }
        }
        pp[k] = p;
        qq[k] = q;
        cs[k] = c;
        sn[k] = s;
      }
      __syncthreads();
      // rows p, q of A
      for (int e = tid; e < npair * n; e += NT) {
        const int k = e / n, col = e % n;
        const int p = pp[k], q = qq[k];
        if (q >= n || sn[k] == 0.0) continue;
        const double c = cs[k], s = sn[k];
        const double x = A[p + col * n], y = A[q + col * n];
        A[p + col * n] = c * x - s * y;
        A[q + col * n] = s * x + c * y;
      }
      __syncthreads();
      // columns p, q of A and of C
      for (int e = tid; e < npair * n; e += NT) {
        const int k = e / n, row = e % n;
        const int p = pp[k], q = qq[k];
        if (q >= n || sn[k] == 0.0) continue;
        const double c = cs[k], s = sn[k];
        const double x = A[row + p * n], y = A[row + q * n];
        A[row + p * n] = c * x - s * y;
        A[row + q * n] = s * x + c * y;
        const double u = C[row + p * n], v = C[row + q * n];
        C[row + p * n] = c * u - s * v;
        C[row + q * n] = s * u + c * v;
      }
      __syncthreads();
    }
  }
  // ascending order, ties by index
  for (int i = tid; i < n; i += NT) {
    const double ai = A[i + i * n];
    int rk = 0;
    for (int j = 0; j < n; ++j) {
      const double aj = A[j + j * n];
      rk += (aj < ai || (aj == ai && j < i)) ? 1 : 0;
    }
    rank[i] = rk;
  }
  __syncthreads();
  for (int e = tid; e < n * n; e += NT) {
    const int r = e % n, c = e / n;
    T[r + rank[c] * n] = C[e];
  }
  for (int i = tid; i < n; i += NT) M.eig[rank[i]] = A[i + i * n];
  __syncthreads();
  for (int e = tid; e < n * n; e += NT) C[e] = T[e];
  __syncthreads();
  const EigCount cnt{nrot, sweeps};
  if (!density) return cnt;
  // P = 2 C_occ C_occ^T, packed
  const long long mp = (long long)n * (n + 1) / 2;
  for (long long q = tid; q < mp; q += NT) {
    int r = (int)((sqrt(8.0 * (double)q + 1.0) - 1.0) * 0.5);
    while ((long long)(r + 1) * (r + 2) / 2 <= q) ++r;
    while ((long long)r * (r + 1) / 2 > q) --r;
    const int c = (int)(q - (long long)r * (r + 1) / 2);
    double s = 0.0;
    for (int k = 0; k < M.nocc; ++k) s += C[r + k * n] * C[c + k * n];
    M.p[q] = 2.0 * s;
  }
  return cnt;
}

template <int NT>
__global__ __launch_bounds__(NT) void k_beig(const BatchMol* __restrict__ mols, const int* __restrict__ do_eig,
                                             BatchState* __restrict__ st, const int* __restrict__ list,
                                             double tol) {
  const int m = list[blockIdx.x];
  if (!do_eig[m]) return;
  const bool warm = st[m].have_c != 0;
  eig_done(mols[m], st[m], beig_global<NT>(mols[m], mols[m].f, warm, tol, st[m].max_sweeps, true), warm);
}

__device__ __forceinline__ int tri(int i) { return (i * (i + 1)) >> 1; }
__device__ __forceinline__ int sym_at(int a, int b) { return a >= b ? tri(a) + b : tri(b) + a; }
// row of packed lower-triangle index e (exact for e < 2^22)
__device__ __forceinline__ int tri_row(int e) {
  int i = (int)((sqrtf(8.0f * (float)e + 1.0f) - 1.0f) * 0.5f);
  if (tri(i + 1) <= e) ++i;
  if (tri(i) > e) --i;
  return i;
}

// Molecules up to kMaxLdsN orbitals are one pair problem of the block-Jacobi
// steps (k_jacobi_step.h), padded to 64 with decoupled large entries: the
// whole eigensolve in one workgroup's LDS, the products with C on the matrix
// cores.  C is 64 x 64 in memory (M.C, identity in the padding).
// A cyclic Jacobi over the packed A, with C beside it in LDS and two barriers
// a round, took 3400 cycles a round at 26 orbitals and 4350 at 60, its chain
// of LDS reads; a round here takes 940 in the level of 32 rounds, and about 1700 with
// the levels between them.
// Larger molecules go to the steps over several workgroups of k_batch_eig.hip.
static_assert(kMaxLdsN == SB, "one pair problem");
constexpr int kLdsThreads = CROSS_THREADS;

__device__ __noinline__ EigCount beig_lds(JacLds& lds, const BatchMol& M, double* f, bool warm, double tol,
                                          int max_sweeps, bool density) {
  const int n = M.n, tid = threadIdx.x;
  __shared__ int rank[SB];
  double(*S)[SB] = lds.s();
  double(*X)[LDSW] = reinterpret_cast<double (*)[LDSW]>(lds.m);
  double(*Y)[LDSW] = reinterpret_cast<double (*)[LDSW]>(lds.m + SB * LDSW);
  double* C = M.C;
  constexpr int PER = SB * SB / kLdsThreads;
  __syncthreads();
  // eigenvectors_LAPACK: F(i,i) += i * 1e-10, in place
  if (tid < n) f[tri(tid) + tid] += (double)(tid + 1) * 1.0e-10;
  __syncthreads();
  auto fp = [&](int r, int c) -> double {
    return r < n && c < n ? f[sym_at(r, c)] : (r == c ? 1.0e4 + r : 0.0);
  };
  d4_t acc[2];
  if (warm) {
    // A = C^T (F C)
#pragma unroll
    for (int it = 0; it < PER; ++it) {
      const int e = tid + kLdsThreads * it;
      X[e % SB][e / SB] = fp(e % SB, e / SB);
      Y[e % SB][e / SB] = C[e];
    }
    __syncthreads();
    acc[0] = acc[1] = d4_t{0.0, 0.0, 0.0, 0.0};
    mfma_tile64_w8([&](int r, int k) { return X[r][k]; }, [&](int k, int c) { return Y[k][c]; }, SB, acc);
    __syncthreads();
    mfma_tile64_w8_store(acc, [&](int r, int c, double v) { X[r][c] = v; });
    __syncthreads();
    acc[0] = acc[1] = d4_t{0.0, 0.0, 0.0, 0.0};
    mfma_tile64_w8([&](int r, int k) { return Y[k][r]; }, [&](int k, int c) { return X[k][c]; }, SB, acc);
    __syncthreads();
    mfma_tile64_w8_store(acc, [&](int r, int c, double v) { S[r][c] = v; });
  } else {
#pragma unroll
    for (int it = 0; it < PER; ++it) {
      const int e = tid + kLdsThreads * it;
      S[e / SB][e % SB] = fp(e / SB, e % SB);
    }
  }
  __syncthreads();
  const int sweeps =
      pair_solve<true>(lds, 0, 1, true, JacSolve{n, nullptr, nullptr, nullptr, nullptr, tol, 0.0, max_sweeps});
  // ascending order, ties by index; the padding stays where it is
  if (tid < SB) {
    const double d = S[tid][tid];
    int rk = tid;
    if (tid < n) {
      rk = 0;
      for (int j = 0; j < n; ++j) {
        const double o = S[j][j];
        rk += (o < d || (o == d && j < tid)) ? 1 : 0;
      }
      M.eig[rk] = d;
    }
    rank[tid] = rk;
  }
  __syncthreads();
  // C Q in the order of the levels, by rows of C's transpose
  double(*Ct)[SB] = lds.s();
  double(*Q)[LDSW] = lds.q();
#pragma unroll
  for (int it = 0; it < PER; ++it) {
    const int e = tid + kLdsThreads * it, r = e % SB, c = e / SB;
    Ct[c][r] = warm ? C[e] : (r == c ? 1.0 : 0.0);
  }
  __syncthreads();
  if (sweeps > 0) {
    acc[0] = acc[1] = d4_t{0.0, 0.0, 0.0, 0.0};
    mfma_tile64_w8([&](int r, int k) { return Ct[k][r]; }, [&](int k, int c) { return Q[k][c]; }, SB, acc);
    __syncthreads();
    mfma_tile64_w8_store(acc, [&](int r, int c, double v) { X[rank[c]][r] = v; });
  } else {
    double v[PER];
#pragma unroll
    for (int it = 0; it < PER; ++it) v[it] = Ct[(tid + kLdsThreads * it) / SB][(tid + kLdsThreads * it) % SB];
    __syncthreads();
#pragma unroll
    for (int it = 0; it < PER; ++it)
      X[rank[(tid + kLdsThreads * it) / SB]][(tid + kLdsThreads * it) % SB] = v[it];
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < PER; ++it) {
    const int e = tid + kLdsThreads * it;
    C[e] = X[e / SB][e % SB];
  }
  if (density) {
    // P = 2 C_occ C_occ^T, packed
    const int nocc = M.nocc;
    acc[0] = acc[1] = d4_t{0.0, 0.0, 0.0, 0.0};
    mfma_tile64_w8([&](int r, int k) { return k < nocc ? X[k][r] : 0.0; },
                   [&](int k, int c) { return X[k][c]; }, (nocc + 3) & ~3, acc);
    mfma_tile64_w8_store(acc, [&](int r, int c, double v) {
      if (r < n && c <= r) M.p[tri(r) + c] = 2.0 * v;
    });
  }
  return EigCount{sweeps * (n * (n - 1) / 2), sweeps};
}

__global__ __launch_bounds__(kLdsThreads, 4) void k_beig_lds(const BatchMol* __restrict__ mols,
                                                             const int* __restrict__ do_eig,
                                                             BatchState* __restrict__ st,
                                                             const int* __restrict__ list, double tol) {
  __shared__ JacLds lds;
  const int m = list[blockIdx.x];
  if (!do_eig[m]) return;
  const bool warm = st[m].have_c != 0;
  eig_done(mols[m], st[m], beig_lds(lds, mols[m], mols[m].f, warm, tol, st[m].max_sweeps, true), warm);
}

// ---- control, part 3: PL, frontier levels, newdg (iter.F90:1030-1041) -------
__device__ void ctl_post(BatchState& s, const BatchMol& M, double pl) {
  s.pl = pl;
  const int ih = max(M.nocc, 1);
  if (ih < M.n) {
    s.eig_homo = M.eig[ih - 1];
    s.eig_lumo = M.eig[ih];
  }
  const double trans = 0.2;
  s.oknewd = (s.pl < s.sellim) || s.oknewd;
  s.newdg = ((s.pl < trans) && s.oknewd) || s.newdg;
  if (s.pl < trans * 0.3333) s.oknewd = 1;
}

__global__ void k_bctl_post(int nmol, const int* __restrict__ list, const BatchMol* __restrict__ mols, BatchState* __restrict__ st,
                            const int* __restrict__ do_eig, const double* __restrict__ scal) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nmol) return;
  const int m = list[i];
  if (!do_eig[m]) return;
  BatchState s = st[m];
  ctl_post(s, mols[m], scal[2 * m]);
  st[m] = s;
}

// ---- the whole SCF of a molecule in one workgroup ----------------------------
// The Fock build of a small molecule (n <= kMaxLdsN) by the workgroup, from P
// and Pa staged in LDS (ps: 2 tri(n) doubles): four lanes per element of the
// diagonal atom blocks (its Coulomb field over every partner, and the
// one-centre terms), a thread per element between two atoms (its exchange
// sum of at most 16 terms).  No partial sums go through memory, and no wave
// is left with an atom's three or four partners: the row and column passes
// of k_fock.hip, a wave per atom, took 95 thousand cycles at 26 orbitals,
// this takes 20 thousand.
template <int NT>
__device__ void fock_small(const FockArgs& a, const int* atom_of, double* ps) {
  const int n = a.sys.norbs, tid = threadIdx.x, mp = tri(n), numat = a.sys.numat;
  double* pas = ps + mp;
  for (int q = tid; q < mp; q += NT) {
    ps[q] = a.p[q];
    pas[q] = a.pa[q];
  }
  __syncthreads();
  auto pr = [](int u, int v) { return u >= v ? tri(u) + v : tri(v) + u; };
  const double* __restrict__ W = a.sys.w;
  // diagonal blocks: element e is pair ab of atom i
  const int nd = (int)a.sys.wcum[numat - 1] + (a.sys.norb[numat - 1] == 4 ? 10 : 1);
  for (int base = 0; base < nd; base += NT / 4) {
    const int e = base + (tid >> 2), part = tid & 3;
    int i = 0;
    double g = 0.0;
    if (e < nd) {
      // the last atom whose first element is not after e
      int lo = 0, hi = numat - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (a.sys.wcum[mid] <= e) lo = mid;
        else hi = mid - 1;
      }
      i = lo;
      const int ab = e - (int)a.sys.wcum[i], limi = a.sys.norb[i] == 4 ? 10 : 1;
      for (int j = part; j < numat; j += 4) {
        if (j == i) continue;
        const int fj = a.sys.nf0[j], nj = a.sys.norb[j], limj = nj == 4 ? 10 : 1;
        // element (ab of i, cd of j) of the pair's block
        const double* wb;
        int step;
        if (j < i) {
          wb = W + a.sys.woff[i] + (long long)limi * a.sys.wcum[j] + ab * limj;
          step = 1;
        } else {
          wb = W + a.sys.woff[j] + (long long)limj * a.sys.wcum[i] + ab;
          step = limi;
        }
        if (nj == 4) {
          double w[10];
#pragma unroll
          for (int cd = 0; cd < 10; ++cd) w[cd] = wb[cd * step];
#pragma unroll
          for (int cd = 0; cd < 10; ++cd) {
            const int x = c_pa[cd], y = c_pb[cd];
            g += w[cd] * ps[tri(fj + x) + fj + y] * (x == y ? 1.0 : 2.0);
          }
        } else {
          g += wb[0] * ps[tri(fj) + fj];
        }
      }
    }
    g += __shfl_xor(g, 1, 64);
    g += __shfl_xor(g, 2, 64);
    if (e < nd && part == 0) {
      const int ab = e - (int)a.sys.wcum[i], ni = a.sys.norb[i], fi = a.sys.nf0[i], lim = ni == 4 ? 10 : 1;
      const int x = c_pa[ab], y = c_pb[ab];
      // one-centre terms (fock1.F90:38-88)
      const double* __restrict__ w1 = W + a.sys.w1off[i];
      for (int k = 0; k < ni; ++k)
        for (int l = 0; l < ni; ++l) {
          const int q = sym_at(fi + k, fi + l);
          g += ps[q] * w1[pr(k, l) * lim + ab] - pas[q] * w1[pr(l, x) * lim + pr(k, y)];
        }
      const int q = tri(fi + x) + fi + y;
      a.f[q] = finit(a, q, x == y) + g;
    }
  }
  // elements between two atoms
  for (int q = tid; q < mp; q += NT) {
    const int r = tri_row(q), c = q - tri(r);
    const int i = atom_of[r], j = atom_of[c];
    if (i == j) continue;
    const int fi = a.sys.nf0[i], fj = a.sys.nf0[j], ni = a.sys.norb[i], nj = a.sys.norb[j];
    const int x = r - fi, u = c - fj, limi = ni == 4 ? 10 : 1, limj = nj == 4 ? 10 : 1;
    const double* __restrict__ wb = W + a.sys.woff[i] + (long long)limi * a.sys.wcum[j];
    double k = 0.0;
    for (int y = 0; y < ni; ++y) {
      const double* row = wb + pr(x, y) * limj;
      const double* pa = pas + tri(fi + y) + fj;
      if (nj == 4) {
#pragma unroll
        for (int v = 0; v < 4; ++v) k += pa[v] * row[pr(u, v)];
      } else {
        k += pa[0] * row[0];
      }
    }
    a.f[q] = finit(a, q, false) - k;
  }
}

// Column pass of the Fock build for atom j by one wave (k_fock.hip has the
// workgroup form).
__device__ void fock_cols_wave(const FockArgs& a, const int j, const int lane) {
  const int nj = a.sys.norb[j];
  const int lim = (nj == 4) ? 10 : 1;
  const long long fj = a.sys.nf0[j];
  const int m = (a.sys.numat - 1 - j) * lim;
  const double* __restrict__ src = a.jcol + a.sys.ccol[j];
  double s = 0.0;
  if (lim == 10) {
    if (lane < 60)
      for (int idx = lane; idx < m; idx += 60) s += src[idx];
    // the six lanes of pair index lane % 10
    double t = s;
#pragma unroll
    for (int k = 1; k < 6; ++k) t += __shfl(s, lane + 10 * k, 64);
    s = t;
  } else {
    for (int idx = lane; idx < m; idx += 64) s += src[idx];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  }
  if (lane >= lim) return;
  const int x = c_pa[lane], y = c_pb[lane];
  // one-centre terms (fock1.F90:38-88)
  const double* __restrict__ w1 = a.sys.w + a.sys.w1off[j];
  auto pr = [](int u, int v) { return u >= v ? u * (u + 1) / 2 + v : v * (v + 1) / 2 + u; };
  double g = 0.0;
  for (int k = 0; k < nj; ++k)
    for (int l = 0; l < nj; ++l) {
      const long long q = pk(fj + k, fj + l);
      g += a.p[q] * w1[pr(k, l) * lim + lane] - a.pa[q] * w1[pr(l, x) * lim + pr(k, y)];
    }
  const long long q = pk(fj + x, fj + y);
  a.f[q] = finit(a, q, x == y) + a.jrow[(long long)j * 10 + lane] + s + g;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ double wave_fmax(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}

// cnvg's diagonal steps (src/SCF/cnvg.F90:16-145, as in k_fock.hip) by one
// wave; returns PL and the extrapolation factor.
__device__ double2 cnvg_diag_wave(int n, double* __restrict__ pnew, double* __restrict__ pold,
                                  double* __restrict__ p1, int niter, int lane) {
  const double rhfuhf = 2.0;
  const double damp = (niter > 3) ? 0.05 : 1.0e10;
  const bool extrap = (niter % 3) != 0;
  double sum1 = 0.0, pl = 0.0, faca = 0.0, facb = 0.0;
  for (int i = lane; i < n; i += 64) {
    const int k = tri(i) + i;
    const double a = pnew[k], o = pold[k];
    sum1 += a;
    const double sa = fabs(a - o);
    pl = fmax(pl, sa);
    if (!extrap) {
      faca += sa * sa;
      const double t = a - 2.0 * o + p1[i];
      facb += t * t;
    }
    p1[i] = o;
    pold[k] = a;
  }
  sum1 = wave_sum(sum1);
  pl = wave_fmax(pl);
  faca = wave_sum(faca);
  facb = wave_sum(facb);
  double fac = 0.0;
  if (facb > 1.0e-10 && faca < 100.0 * facb) fac = sqrt(faca / facb);
  double sum2 = 0.0;
  for (int i = lane; i < n; i += 64) {
    const int k = tri(i) + i;
    double v = pold[k];
    const double o = p1[i];
    if (fabs(v - o) > damp) v = o + ((v - o) >= 0.0 ? damp : -damp);
    else v = v + fac * (v - o);
    v = fmin(rhfuhf, fmax(v, 0.0));
    pold[k] = v;
    pnew[k] = v;
    sum2 += v;
  }
  sum2 = wave_sum(sum2);
  const double sum0 = sum1;
  for (int it = 0; it < 1000; ++it) {
    const double sc = (sum2 > 1.0e-3) ? sum1 / sum2 : 0.0;
    sum1 = sum0;
    if (sum2 < 1.0e-3 || fabs(sc - 1.0) < 1.0e-5) break;
    double s2 = 0.0, nclamp = 0.0;
    for (int i = lane; i < n; i += 64) {
      const int k = tri(i) + i;
      double v = fmax(pold[k] * sc + 1.0e-20, 0.0);
      if (v > rhfuhf) {
        v = rhfuhf;
        nclamp += 1.0;
      } else {
        s2 += v;
      }
      pold[k] = v;
      pnew[k] = v;
    }
    sum2 = wave_sum(s2);
    sum1 -= rhfuhf * wave_sum(nclamp);
  }
  return make_double2(pl, fac);
}

// The SCF of molecule list[blockIdx.x] (entry 0 without a list), from the
// state and densities in memory until it is done or `cap` Fock builds have
// run.  No molecule waits for another: in lockstep, a launch per phase over
// all molecules, every iteration took the longest eigensolve of its size
// class and twenty launches, and 64 molecules took 109 ms where they now take
// 13 (400: 137 -> 23, 4096: 403 -> 213).  With M.fexit, a finished molecule is
// diagonalized once more to 1e-12, as iter does at its exit, and phase_lock'ed
// if asked.
template <int NT, bool LDS>
__device__ __forceinline__ void scf_body(JacLds* lds, const FockArgs* __restrict__ args,
                                         const BatchMol* __restrict__ mols, BatchState* __restrict__ st,
                                         const int* __restrict__ list, double tol, int cap, int lock) {
  constexpr int NW = NT / 64;
  __shared__ BatchState s;
  __shared__ double red[NW];
  __shared__ double2 plfac;
  const int m = list ? list[blockIdx.x] : 0;
  const BatchMol M = mols[m];
  FockArgs a = args[m];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, n = M.n;
  auto eig = [&](double* f, bool warm, double t, bool density) {
    if constexpr (LDS) return beig_lds(*lds, M, f, warm, t, s.max_sweeps, density);
    else return beig_global<NT>(M, f, warm, t, s.max_sweeps, density);
  };
  if (tid == 0) s = st[m];
  __shared__ int atom_of[kMaxLdsN];
  if constexpr (LDS)
    for (int i = tid; i < M.numat; i += NT)
      for (int k = 0; k < a.sys.norb[i]; ++k) atom_of[a.sys.nf0[i] + k] = i;
  __syncthreads();
  for (int pass = 0; pass < cap; ++pass) {
    if (s.done) break;
    __syncthreads();
    if (tid == 0) ctl_pre(s);
    __syncthreads();
    a.init_mode = s.mode;
    a.shift = s.shift;
    if constexpr (LDS) {
      fock_small<NT>(a, atom_of, lds->m);
    } else {
      for (int i = M.numat - 1 - w; i >= 0; i -= NW) fock_rows_body<64>(a, i, lane);
      __syncthreads();
      for (int j = w; j < M.numat; j += NW) fock_cols_wave(a, j, lane);
    }
    __syncthreads();
    double e = 0.0;
    for (int r = w; r < n; r += NW)
      for (int c = lane; c <= r; c += 64) {
        const int q = tri(r) + c;
        const double v = a.pa[q] * (a.h[q] + a.f[q]);
        e += (c == r) ? 0.5 * v : v;
      }
    e = wave_sum(e);
    if (lane == 0) red[w] = e;
    __syncthreads();
    if (tid == 0) {
      e = red[0];
      for (int i = 1; i < NW; ++i) e += red[i];
      ctl_mid(s, 2.0 * e);
    }
    __syncthreads();
    if (s.done) break;
    if (!s.do_eig) continue;
    const bool warm = s.have_c != 0;
    double t = tol;
    if (s.adaptive && s.pl > 10.0 * s.pltest) t = fmax(tol, fmin(1.0e-5, 1.0e-3 * s.pl));
    const EigCount cnt = eig(M.f, warm, t, true);
    __syncthreads();
    eig_done(M, s, cnt, warm);
    if (w == 0) {
      const double2 r = cnvg_diag_wave(n, M.p, M.pold, M.p1, s.niter, lane);
      if (lane == 0) plfac = r;
    }
    __syncthreads();
    const double fac = plfac.y;
    for (int r = w; r < n; r += NW)
      for (int c = lane; c <= r; c += 64) {
        const int q = tri(r) + c;
        double v = M.p[q];
        if (c < r) {
          v += fac * (v - M.pold[q]);
          M.pold[q] = v;
          M.p[q] = v;
        }
        M.pa[q] = 0.5 * v;
      }
    if (tid == 0) ctl_post(s, M, plfac.x);
    __syncthreads();
  }
  if (M.fexit && s.done && isfinite(s.ee)) {
    for (int q = tid; q < tri(n); q += NT) M.fexit[q] = M.f[q];
    __syncthreads();
    const bool warm = s.have_c != 0;
    const EigCount cnt = eig(M.fexit, warm, 1.0e-12, false);
    __syncthreads();
    eig_done(M, s, cnt, warm);
    if (lock) {
      // the largest coefficient of each column positive (the first of equals)
      for (int col = w; col < n; col += NW) {
        double* v = M.C + (size_t)col * (LDS ? SB : n);
        double best = 0.0, sgn = 0.0;
        int bi = n;
        for (int r = lane; r < n; r += 64) {
          const double x = fabs(v[r]);
          if (x > best) { best = x; sgn = v[r]; bi = r; }
        }
        for (int o = 32; o > 0; o >>= 1) {
          const double b2 = __shfl_xor(best, o, 64), s2 = __shfl_xor(sgn, o, 64);
          const int i2 = __shfl_xor(bi, o, 64);
          if (b2 > best || (b2 == best && i2 < bi)) { best = b2; sgn = s2; bi = i2; }
        }
        if (sgn < 0.0)
          for (int r = lane; r < n; r += 64) v[r] = -v[r];
      }
    }
  }
  __syncthreads();
  if (tid == 0) st[m] = s;
}

__global__ __launch_bounds__(kLdsThreads, 4) void k_bscf_lds(const FockArgs* __restrict__ args,
                                                             const BatchMol* __restrict__ mols,
                                                             BatchState* __restrict__ st,
                                                             const int* __restrict__ list, double tol, int cap,
                                                             int lock) {
  __shared__ JacLds lds;
  scf_body<kLdsThreads, true>(&lds, args, mols, st, list, tol, cap, lock);
}

template <int NT>
__global__ __launch_bounds__(NT) void k_bscf(const FockArgs* __restrict__ args, const BatchMol* __restrict__ mols,
                                             BatchState* __restrict__ st, const int* __restrict__ list, double tol,
                                             int cap, int lock) {
  scf_body<NT, false>(nullptr, args, mols, st, list, tol, cap, lock);
}

// The starting densities (iter.F90:269-300): P the atoms' diagonal, Pa its
// share of one spin, the previous density and diagonal those of Pa.
__global__ __launch_bounds__(256) void k_binit(const BatchMol* __restrict__ mols, const double* __restrict__ pdiag,
                                               const long long* __restrict__ orb_off, int* __restrict__ act,
                                               int* __restrict__ do_eig) {
  const BatchMol M = mols[blockIdx.x];
  if (threadIdx.x == 0) act[blockIdx.x] = do_eig[blockIdx.x] = 0;
  const double* d = pdiag + orb_off[blockIdx.x];
  const double w1 = M.nocc / (M.nocc + 1.0e-6 + M.nocc), share = w1 < 1e-6 ? 0.5 : w1;
  for (int q = threadIdx.x; q < tri(M.n); q += 256) {
    const int r = tri_row(q);
    const double v = q == tri(r) + r ? d[r] : 0.0;
    M.p[q] = v;
    M.pa[q] = M.pold[q] = v * share;
  }
  for (int i = threadIdx.x; i < M.n; i += 256) M.p1[i] = d[i] * share;
}

// Pa = P / 2 for the molecules that stepped
__global__ __launch_bounds__(256) void k_bhalf(const BatchMol* __restrict__ mols, const int* __restrict__ blk_mol,
                                               const int* __restrict__ blk_row, const int* __restrict__ do_eig) {
  const int m = blk_mol[blockIdx.x];
  if (!do_eig[m]) return;
  const BatchMol& M = mols[m];
  const long long r = blk_row[blockIdx.x];
  for (long long c = threadIdx.x; c <= r; c += 256) {
    const long long q = r * (r + 1) / 2 + c;
    M.pa[q] = 0.5 * M.p[q];
  }
}

inline int cdiv(long long a, long long b) { return (int)((a + b - 1) / b); }

}  // namespace
}  // namespace mhip

using namespace mhip;

struct mhip_batch {
  int nmol = 0;
  hipStream_t s = nullptr;
  std::vector<int> n_h, nocc_h, numat_h;
  // device storage
  DevBuf w, h, f, p, pa, pold, p1, C, eig, jrow, jcol;
  std::vector<BatchMol> mol_h;  // as mols has them
  DevBuf global;                // the matrices of the global-memory form, once it is asked for
  DevBuf nf0, norb, woff, wcum, w1off, ccol, heavy, light, nhb, nlb;
  DevBuf args, mols, cnv, st, act, doeig, mode, niter, shift, ee, partial, scal, orboff;
  DevBuf pdiag, st0;  // starting diagonals and control states, where every run begins
  int device = 0;  // that everything here belongs to
  // a stream and an event per size class that runs a workgroup to a molecule:
  // the classes fill each other's tails
  hipStream_t cs[4] = {};
  hipEvent_t ev[5] = {};
  DevBuf atom_mol, atom_idx, row_mol, row_idx;
  int n_atom_blk = 0, n_row_blk = 0;
  // molecules by eigensolver class (workgroup size), in launch order
  std::vector<int> cls_count, cls_nmax;
  BatchJacobi* bj = nullptr;         // the classes above kMaxLdsN
  int small_atoms = 0, small_rows = 0;  // workgroups of the others in the atom and row lists, which they begin
  bool force_global_eig = false;
  DevBuf cls_list;
  int tile[4] = {64, 128, 256, 256};   // workgroup size per class (n <= 32, 64, 128, 256)
  double tol = 1.0e-10;
  int max_sweeps = kEigSweeps;
  std::vector<BatchState> init_state;
  // eager timing of the eigensolver launches per size class
  hipEvent_t eig_ev[4][2] = {};
  bool eig_timing = false;
};

namespace {

int size_class(int n) { return n <= 32 ? 0 : (n <= 64 ? 1 : (n <= 128 ? 2 : 3)); }

// fn(std::integral_constant<int, NT>) for the workgroup size `tile`
template <class F>
void with_tile(int tile, F&& fn) {
  switch (tile) {
    case 64: fn(std::integral_constant<int, 64>()); break;
    case 128: fn(std::integral_constant<int, 128>()); break;
    case 512: fn(std::integral_constant<int, 512>()); break;
    case 1024: fn(std::integral_constant<int, 1024>()); break;
    default: fn(std::integral_constant<int, 256>()); break;
  }
}

// Classes 0 and 1 in LDS, a workgroup to a molecule; with the matrices in
// memory (the comparison form) every class.
void launch_eig_class(mhip_batch* b, int cls, int offset, int count) {
  if (count <= 0) return;
  auto* mols = b->mols.as<BatchMol>();
  auto* st = b->st.as<BatchState>();
  const int* list = b->cls_list.as<int>() + offset;
  const int* de = b->doeig.as<int>();
  if (!b->force_global_eig)
    hipLaunchKernelGGL(k_beig_lds, dim3(count), dim3(kLdsThreads), 0, b->s, mols, de, st, list, b->tol);
  else
    with_tile(b->tile[cls], [&](auto nt) {
      constexpr int NT = decltype(nt)::value;
      hipLaunchKernelGGL(k_beig<NT>, dim3(count), dim3(NT), 0, b->s, mols, de, st, list, b->tol);
    });
  MHIP_LAUNCH_CHECK();
}

void launch_scf_class(mhip_batch* b, hipStream_t s, int cls, int offset, int cap) {
  auto* args = b->args.as<FockArgs>();
  auto* mols = b->mols.as<BatchMol>();
  auto* st = b->st.as<BatchState>();
  const int* list = b->cls_list.as<int>() + offset;
  const int n = b->cls_count[cls];
  if (!b->force_global_eig)
    hipLaunchKernelGGL(k_bscf_lds, dim3(n), dim3(kLdsThreads), 0, s, args, mols, st, list, b->tol, cap, 0);
  else
    with_tile(b->tile[cls], [&](auto nt) {
      constexpr int NT = decltype(nt)::value;
      hipLaunchKernelGGL(k_bscf<NT>, dim3(n), dim3(NT), 0, s, args, mols, st, list, b->tol, cap, 0);
    });
  MHIP_LAUNCH_CHECK();
}

// For the first n classes, where they have a molecule.
void ensure_class_streams(mhip_batch* b, int n) {
  for (int c = 0; c < n; ++c) {
    if (b->cls_count[c] == 0) continue;
    if (!b->cs[c]) MHIP_CHECK(hipStreamCreateWithFlags(&b->cs[c], hipStreamNonBlocking));
    if (!b->ev[c]) MHIP_CHECK(hipEventCreateWithFlags(&b->ev[c], hipEventDisableTiming));
  }
}

// A and T of every molecule, and C of those that have none in the default form,
// for the form with its matrices in memory.  They are left out until it is
// chosen: 3 n^2 beside the 4 npad^2 that the block-Jacobi form works in.
void ensure_global_form(mhip_batch* b) {
  if (b->global.ptr) return;
  struct OnDevice {
    int before = 0;
    explicit OnDevice(int device) {
      MHIP_CHECK(hipGetDevice(&before));
      MHIP_CHECK(hipSetDevice(device));
    }
    ~OnDevice() { (void)hipSetDevice(before); }
  } on(b->device);
  ensure_class_streams(b, 4);
  size_t len = 0;
  for (const BatchMol& q : b->mol_h) len += (size_t)q.n * q.n * (q.C ? 2 : 3);
  b->global.ensure(sizeof(double) * len);
  double* at = b->global.as<double>();
  for (BatchMol& q : b->mol_h) {
    const size_t sz = (size_t)q.n * q.n;
    q.A = at;
    q.T = at + sz;
    at += 2 * sz;
    if (q.C) continue;
    q.C = at;
    at += sz;
  }
  MHIP_CHECK(hipMemcpy(b->mols.ptr, b->mol_h.data(), sizeof(BatchMol) * b->nmol, hipMemcpyHostToDevice));
}

// One iteration of every molecule (the eigensolver profile), or of those of
// the block-Jacobi classes alone (big_only), a launch per phase over all of
// them; returns how many of the latter are not done.
int one_iteration(mhip_batch* b, bool big_only) {
  hipStream_t s = b->s;
  const int l0 = big_only ? b->cls_count[0] + b->cls_count[1] : 0, nm = b->nmol - l0;
  const int a0 = big_only ? b->small_atoms : 0, na = b->n_atom_blk - a0;
  const int r0 = big_only ? b->small_rows : 0, nr = b->n_row_blk - r0;
  const int* list = b->cls_list.as<int>() + l0;
  const int* row_mol = b->row_mol.as<int>() + r0;
  const int* row_idx = b->row_idx.as<int>() + r0;
  const int cb = cdiv(nm, 64);
  hipLaunchKernelGGL(k_bctl_pre, dim3(cb), dim3(64), 0, s, nm, list, b->st.as<BatchState>(), b->act.as<int>(),
                     b->mode.as<int>(), b->niter.as<int>(), b->shift.as<double>());
  MHIP_LAUNCH_CHECK();
  fock_build_batch(s, b->args.as<FockArgs>(), na, b->atom_mol.as<int>() + a0, b->atom_idx.as<int>() + a0,
                   b->act.as<int>(), b->mode.as<int>(), b->shift.as<double>());
  helect_batch(s, b->args.as<FockArgs>(), b->nmol, nr, row_mol, row_idx, b->act.as<int>(),
               b->orboff.as<long long>(), b->partial.as<double>(), 2.0, b->ee.as<double>());
  hipLaunchKernelGGL(k_bctl_mid, dim3(cb), dim3(64), 0, s, nm, list, b->st.as<BatchState>(), b->ee.as<double>(),
                     b->doeig.as<int>());
  MHIP_LAUNCH_CHECK();
  int open = 0, off = 0;
  for (int c = big_only ? 2 : 0; c < 4; ++c) {
    if (b->eig_timing) MHIP_CHECK(hipEventRecord(b->eig_ev[c][0], s));
    if (c < 2 || b->force_global_eig) launch_eig_class(b, c, off, b->cls_count[c]);
    else if (b->bj && (!big_only || c == 2))
      // by itself only for its own time
      open += bj_solve(b->bj, s, b->st.as<BatchState>(), b->doeig.as<int>(), b->tol, b->max_sweeps,
                       big_only || c == 2 ? 128 : 192, !big_only && c == 2 ? 128 : 256);
    if (b->eig_timing) MHIP_CHECK(hipEventRecord(b->eig_ev[c][1], s));
    off += b->cls_count[c];
  }
  if (big_only && open == 0) return 0;
  cnvg_batch(s, b->cnv.as<BatchCnvg>(), b->nmol, nr, row_mol, row_idx, b->doeig.as<int>(), b->niter.as<int>(),
             b->scal.as<double>());
  hipLaunchKernelGGL(k_bctl_post, dim3(cb), dim3(64), 0, s, nm, list, b->mols.as<BatchMol>(), b->st.as<BatchState>(),
                     b->doeig.as<int>(), b->scal.as<double>());
  MHIP_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_bhalf, dim3(nr), dim3(256), 0, s, b->mols.as<BatchMol>(), row_mol, row_idx,
                     b->doeig.as<int>());
  MHIP_LAUNCH_CHECK();
  return open;
}

template <class F>
int bguard(F&& fn) {
  try {
    fn();
    return 0;
  } catch (const HipError& e) {
    set_error(e.msg);
    return 1;
  }
}

}  // namespace

namespace mhip {

BatchState batch_start(double enuclr, double atheat, double scfcrt, int itrmax) {
  BatchState z{};
  z.itrmax = itrmax > 0 ? itrmax : 2000;
  z.max_sweeps = kEigSweeps;
  z.ten = -80.0;
  z.shift = 1.0;
  z.shfmax = 20.0;
  z.pl = 1.0;
  z.eold = 100.0;
  z.iredy = 1;
  z.enuclr = enuclr;
  z.atheat = atheat;
  const double scf = std::max(scfcrt > 0 ? scfcrt : 1.0e-4, 1e-12);
  z.selcon = std::min(std::min(scf * 100.0, 0.1), scf);
  z.pltest = 0.05 * std::sqrt(std::fabs(z.selcon));
  return z;
}

bool scf_one_workgroup(hipStream_t s, int n, const FockArgs* args, const BatchMol* mol, BatchState* st, double tol,
                       int phase_lock) {
  if (n > kMaxLdsN) return false;
  hipLaunchKernelGGL(k_bscf_lds, dim3(1), dim3(kLdsThreads), 0, s, args, mol, st, nullptr, tol, INT_MAX, phase_lock);
  MHIP_LAUNCH_CHECK();
  return true;
}

}  // namespace mhip

extern "C" {

int mhip_batch_create(int nmol, const mhip_batch_molecule* mols, mhip_batch** out) {
  return bguard([&] {
    MHIP_REQUIRE(nmol > 0 && mols && out, "mhip_batch_create: bad arguments");
    auto* b = new mhip_batch();
    b->nmol = nmol;
    MHIP_CHECK(hipStreamCreateWithFlags(&b->s, hipStreamNonBlocking));
    MHIP_CHECK(hipGetDevice(&b->device));
    MHIP_CHECK(hipEventCreateWithFlags(&b->ev[4], hipEventDisableTiming));
    // ---- host tables, then one upload per array
    std::vector<long long> o_w(nmol), o_mp(nmol), o_nn(nmol), o_n(nmol), o_at(nmol), o_cc(nmol);
    long long tw = 0, tmp = 0, tnn = 0, tn = 0, tat = 0, tcc = 0;
    std::vector<int> nf0_all, norb_all, heavy_all, light_all, nhb_all, nlb_all;
    std::vector<long long> woff_all, wcum_all, w1off_all, ccol_all;
    for (int m = 0; m < nmol; ++m) {
      const mhip_batch_molecule& M = mols[m];
      const int n = M.norbs, na = M.numat;
      MHIP_REQUIRE(n > 0 && n <= kMaxBatchN && na > 0, "mhip_batch_create: molecule size out of range (n <= 256)");
      MHIP_REQUIRE(M.nclose >= 0 && M.nclose <= n, "mhip_batch_create: bad nclose");
      b->n_h.push_back(n);
      b->nocc_h.push_back(M.nclose);
      b->numat_h.push_back(na);
      o_w[m] = tw;
      o_mp[m] = tmp;
      o_nn[m] = tnn;
      o_n[m] = tn;
      o_at[m] = tat;
      o_cc[m] = tcc;
      // atom-pair tables (the same construction as the single-system upload)
      long long kr = 0, wc = 0, cc = 0;
      int nh = 0, nl = 0;
      for (int i = 0; i < na; ++i) {
        const int f0 = M.nfirst[i] - 1, no = M.nlast[i] - M.nfirst[i] + 1;
        MHIP_REQUIRE(no == 1 || no == 4, "mhip_batch_create: only s and sp atoms");
        MHIP_REQUIRE(i == 0 ? f0 == 0 : f0 == nf0_all.back() + norb_all.back(),
                     "mhip_batch_create: orbitals must be contiguous by atom");
        nf0_all.push_back(f0);
        norb_all.push_back(no);
        const int lim = no * (no + 1) / 2;
        woff_all.push_back(kr);
        wcum_all.push_back(wc);
        kr += (long long)lim * wc;
        w1off_all.push_back(kr);
        kr += (long long)lim * lim;
        wc += lim;
        nhb_all.push_back(nh);
        nlb_all.push_back(nl);
        if (no == 4) { heavy_all.push_back(i); ++nh; } else { light_all.push_back(i); ++nl; }
        ccol_all.push_back(cc);
        cc += (long long)(na - 1 - i) * lim;
      }
      MHIP_REQUIRE(kr == M.n2elec, "mhip_batch_create: n2elec does not match the hcore layout");
      MHIP_REQUIRE(nf0_all.back() + norb_all.back() == n, "mhip_batch_create: nlast(numat) != norbs");
      tw += kr;
      tmp += (long long)n * (n + 1) / 2;
      if (n <= kMaxLdsN) tnn += SB * SB;  // C, padded
      tn += n;
      tat += na;
      tcc += std::max(cc, 1LL);
    }
    // heavy/light lists hold indices within each molecule: offsets per molecule
    std::vector<long long> o_heavy(nmol), o_light(nmol);
    {
      long long hh = 0, ll = 0;
      for (int m = 0; m < nmol; ++m) {
        o_heavy[m] = hh;
        o_light[m] = ll;
        for (int i = 0; i < mols[m].numat; ++i) {
          if (mols[m].nlast[i] - mols[m].nfirst[i] == 3) ++hh; else ++ll;
        }
      }
    }
    hipStream_t s = b->s;
    b->w.ensure(sizeof(double) * std::max(tw, 1LL));
    b->h.ensure(sizeof(double) * tmp);
    for (DevBuf* x : {&b->f, &b->p, &b->pa, &b->pold}) x->ensure(sizeof(double) * tmp);
    b->p1.ensure(sizeof(double) * tn);
    b->eig.ensure(sizeof(double) * tn);
    b->C.ensure(sizeof(double) * std::max(tnn, 1LL));
    b->jrow.ensure(sizeof(double) * 10 * tat);
    b->jcol.ensure(sizeof(double) * tcc);
    for (int m = 0; m < nmol; ++m) {
      const mhip_batch_molecule& M = mols[m];
      const long long mp = (long long)M.norbs * (M.norbs + 1) / 2;
      if (M.n2elec)
        MHIP_CHECK(hipMemcpyAsync(b->w.as<double>() + o_w[m], M.w, sizeof(double) * M.n2elec,
                                  hipMemcpyHostToDevice, s));
      MHIP_CHECK(hipMemcpyAsync(b->h.as<double>() + o_mp[m], M.h, sizeof(double) * mp, hipMemcpyHostToDevice, s));
    }
    auto upv = [&](DevBuf& d, const void* src, size_t bytes) {
      d.ensure(bytes ? bytes : 8);
      if (bytes) MHIP_CHECK(hipMemcpyAsync(d.ptr, src, bytes, hipMemcpyHostToDevice, s));
    };
    upv(b->nf0, nf0_all.data(), sizeof(int) * nf0_all.size());
    upv(b->norb, norb_all.data(), sizeof(int) * norb_all.size());
    upv(b->woff, woff_all.data(), sizeof(long long) * woff_all.size());
    upv(b->wcum, wcum_all.data(), sizeof(long long) * wcum_all.size());
    upv(b->w1off, w1off_all.data(), sizeof(long long) * w1off_all.size());
    upv(b->ccol, ccol_all.data(), sizeof(long long) * ccol_all.size());
    upv(b->heavy, heavy_all.data(), sizeof(int) * heavy_all.size());
    upv(b->light, light_all.data(), sizeof(int) * light_all.size());
    upv(b->nhb, nhb_all.data(), sizeof(int) * nhb_all.size());
    upv(b->nlb, nlb_all.data(), sizeof(int) * nlb_all.size());
    // molecules grouped by eigensolver class
    std::vector<int> order;
    b->cls_count.assign(4, 0);
    b->cls_nmax.assign(4, 0);
    for (int c = 0; c < 4; ++c)
      for (int m = 0; m < nmol; ++m)
        if (size_class(b->n_h[m]) == c) {
          order.push_back(m);
          b->cls_count[c]++;
          b->cls_nmax[c] = std::max(b->cls_nmax[c], b->n_h[m]);
        }
    ensure_class_streams(b, 2);
    // the largest of each class first: they take the longest
    for (int c = 0, o = 0; c < 4; o += b->cls_count[c++])
      std::stable_sort(order.begin() + o, order.begin() + o + b->cls_count[c],
                       [&](int x, int y) { return b->n_h[x] > b->n_h[y]; });
    // per-molecule argument blocks
    std::vector<FockArgs> args(nmol);
    std::vector<BatchMol>& bm = b->mol_h;
    bm.resize(nmol);
    std::vector<BatchCnvg> cv(nmol);
    std::vector<long long> orboff(nmol);
    std::vector<int> atom_mol, atom_idx, row_mol, row_idx;
    b->init_state.resize(nmol);
    std::vector<double> pdiag;
    for (int m = 0; m < nmol; ++m) {
      const mhip_batch_molecule& M = mols[m];
      const int n = M.norbs;
      FockArgs& a = args[m];
      a.sys.numat = M.numat;
      a.sys.norbs = n;
      a.sys.n2elec = M.n2elec;
      a.sys.nf0 = b->nf0.as<int>() + o_at[m];
      a.sys.norb = b->norb.as<int>() + o_at[m];
      a.sys.woff = b->woff.as<long long>() + o_at[m];
      a.sys.wcum = b->wcum.as<long long>() + o_at[m];
      a.sys.w1off = b->w1off.as<long long>() + o_at[m];
      a.sys.ccol = b->ccol.as<long long>() + o_at[m];
      a.sys.heavy = b->heavy.as<int>() + o_heavy[m];
      a.sys.light = b->light.as<int>() + o_light[m];
      a.sys.nheavy_before = b->nhb.as<int>() + o_at[m];
      a.sys.nlight_before = b->nlb.as<int>() + o_at[m];
      a.sys.w = b->w.as<double>() + o_w[m];
      a.h = b->h.as<double>() + o_mp[m];
      a.p = b->p.as<double>() + o_mp[m];
      a.pa = b->pa.as<double>() + o_mp[m];
      a.fin = b->f.as<double>() + o_mp[m];
      a.f = b->f.as<double>() + o_mp[m];
      a.jrow = b->jrow.as<double>() + 10 * o_at[m];
      a.jcol = b->jcol.as<double>() + o_cc[m];
      BatchMol& q = bm[m];
      q.n = n;
      q.nocc = M.nclose;
      q.numat = M.numat;
      q.f = a.f;
      q.p = b->p.as<double>() + o_mp[m];
      q.pa = b->pa.as<double>() + o_mp[m];
      q.pold = b->pold.as<double>() + o_mp[m];
      q.p1 = b->p1.as<double>() + o_n[m];
      q.C = n <= kMaxLdsN ? b->C.as<double>() + o_nn[m] : nullptr;
      q.eig = b->eig.as<double>() + o_n[m];
      cv[m] = BatchCnvg{n, q.p, q.pold, q.p1};
      orboff[m] = o_n[m];
      pdiag.insert(pdiag.end(), M.pdiag, M.pdiag + n);
      b->init_state[m] = batch_start(M.enuclr, M.atheat, M.scfcrt, M.itrmax);
    }
    for (int k = 0; k < nmol; ++k) {
      const int m = order[k];
      if (k == b->cls_count[0] + b->cls_count[1]) {
        b->small_atoms = (int)atom_mol.size();
        b->small_rows = (int)row_mol.size();
      }
      for (int i = 0; i < mols[m].numat; ++i) {
        atom_mol.push_back(m);
        atom_idx.push_back(i);
      }
      for (int r = 0; r < mols[m].norbs; ++r) {
        row_mol.push_back(m);
        row_idx.push_back(r);
      }
    }
    b->n_atom_blk = (int)atom_mol.size();
    b->n_row_blk = (int)row_mol.size();
    upv(b->args, args.data(), sizeof(FockArgs) * nmol);
    upv(b->mols, bm.data(), sizeof(BatchMol) * nmol);
    upv(b->cnv, cv.data(), sizeof(BatchCnvg) * nmol);
    upv(b->orboff, orboff.data(), sizeof(long long) * nmol);
    upv(b->atom_mol, atom_mol.data(), sizeof(int) * atom_mol.size());
    upv(b->atom_idx, atom_idx.data(), sizeof(int) * atom_idx.size());
    upv(b->row_mol, row_mol.data(), sizeof(int) * row_mol.size());
    upv(b->row_idx, row_idx.data(), sizeof(int) * row_idx.size());
    b->st.ensure(sizeof(BatchState) * nmol);
    for (DevBuf* x : {&b->act, &b->doeig, &b->mode, &b->niter}) x->ensure(sizeof(int) * nmol);
    for (DevBuf* x : {&b->shift, &b->ee}) x->ensure(sizeof(double) * nmol);
    b->scal.ensure(sizeof(double) * 2 * nmol);
    b->partial.ensure(sizeof(double) * tn);
    upv(b->pdiag, pdiag.data(), sizeof(double) * tn);
    upv(b->st0, b->init_state.data(), sizeof(BatchState) * nmol);
    upv(b->cls_list, order.data(), sizeof(int) * nmol);
    const std::vector<int> big(order.begin() + b->cls_count[0] + b->cls_count[1], order.end());
    if (!big.empty()) b->bj = bj_create(bm, big);
    MHIP_CHECK(hipStreamSynchronize(s));  // the host vectors go out of scope
    *out = b;
  });
}

int mhip_batch_set_tiles(mhip_batch* b, const int* tiles) {
  return bguard([&] {
    MHIP_REQUIRE(b && tiles, "mhip_batch_set_tiles: bad arguments");
    for (int c = 0; c < 4; ++c) {
      MHIP_REQUIRE(tiles[c] == 64 || tiles[c] == 128 || tiles[c] == 256 || tiles[c] == 512 || tiles[c] == 1024,
                   "mhip_batch_set_tiles: workgroup sizes are 64, 128, 256, 512 or 1024");
      b->tile[c] = tiles[c];
    }
  });
}

int mhip_batch_set_eig_lds(mhip_batch* b, int lds) {
  return bguard([&] {
    MHIP_REQUIRE(b, "mhip_batch_set_eig_lds: bad arguments");
    if (lds == 0) ensure_global_form(b);
    b->force_global_eig = lds == 0;
  });
}

int mhip_batch_set_eig_sweeps(mhip_batch* b, int max_sweeps) {
  return bguard([&] {
    MHIP_REQUIRE(b && max_sweeps > 0 && max_sweeps <= kEigSweeps, "mhip_batch_set_eig_sweeps: 1 to 60 sweeps");
    b->max_sweeps = max_sweeps;
    for (auto& z : b->init_state) z.max_sweeps = max_sweeps;
    MHIP_CHECK(hipMemcpy(b->st0.ptr, b->init_state.data(), sizeof(BatchState) * b->nmol, hipMemcpyHostToDevice));
  });
}

// self-consistent, by levels that every eigensolve on the way converged to
static bool converged(const BatchState& z) { return z.converged && !z.stuck; }

// the per-molecule state and the starting densities, before a run
static void reset_batch(mhip_batch* b) {
  MHIP_CHECK(hipMemcpyAsync(b->st.ptr, b->st0.ptr, sizeof(BatchState) * b->nmol, hipMemcpyDeviceToDevice, b->s));
  hipLaunchKernelGGL(k_binit, dim3(b->nmol), dim3(256), 0, b->s, b->mols.as<BatchMol>(), b->pdiag.as<double>(),
                     b->orboff.as<long long>(), b->act.as<int>(), b->doeig.as<int>());
  MHIP_LAUNCH_CHECK();
}

int mhip_batch_eig_profile(mhip_batch* b, int iters, double* ms, double* flops, long long* rotations) {
  return bguard([&] {
    MHIP_REQUIRE(b && iters > 0 && ms && flops, "mhip_batch_eig_profile: bad arguments");
    hipStream_t s = b->s;
    reset_batch(b);
    for (int c = 0; c < 4; ++c) {
      ms[c] = 0.0;
      flops[c] = 0.0;
      if (rotations) rotations[c] = 0;
      for (int e = 0; e < 2; ++e) MHIP_CHECK(hipEventCreate(&b->eig_ev[c][e]));
    }
    b->eig_timing = true;
    struct Off {
      mhip_batch* b;
      ~Off() {
        b->eig_timing = false;
        for (auto& c : b->eig_ev)
          for (auto& e : c)
            if (e) {
              (void)hipEventDestroy(e);
              e = nullptr;
            }
      }
    } off{b};
    for (int it = 0; it < iters; ++it) {
      one_iteration(b, false);
      MHIP_CHECK(hipStreamSynchronize(s));
      for (int c = 0; c < 4; ++c) {
        float t = 0.0f;
        MHIP_CHECK(hipEventElapsedTime(&t, b->eig_ev[c][0], b->eig_ev[c][1]));
        ms[c] += t;
      }
    }
    std::vector<BatchState> hs(b->nmol);
    MHIP_CHECK(hipMemcpy(hs.data(), b->st.ptr, sizeof(BatchState) * b->nmol, hipMemcpyDeviceToHost));
    for (int m = 0; m < b->nmol; ++m) {
      const int c = size_class(b->n_h[m]);
      flops[c] += hs[m].eig_flops;
      if (rotations) rotations[c] += hs[m].eig_rot;
    }
  });
}

// Run the batched SCF from the starting densities, at most iters_per_graph *
// max_launches iterations (and recomputed Fock builds) of each molecule.
int mhip_batch_run(mhip_batch* b, int iters_per_graph, int max_launches, double* seconds, int* n_converged) {
  return bguard([&] {
    MHIP_REQUIRE(b && iters_per_graph > 0 && max_launches > 0, "mhip_batch_run: bad arguments");
    hipStream_t s = b->s;
    const int cap = (int)std::min<long long>((long long)iters_per_graph * max_launches, 1 << 30);
    reset_batch(b);
    MHIP_CHECK(hipStreamSynchronize(s));
    const auto t0 = std::chrono::steady_clock::now();
    MHIP_CHECK(hipEventRecord(b->ev[4], s));
    // small molecules: each class on a stream of its own, a workgroup for
    // every molecule from start to end; beside them the block-Jacobi classes,
    // an iteration at a time
    const int one_wg = b->force_global_eig ? 4 : 2;
    for (int c = 0, off = 0; c < one_wg; off += b->cls_count[c++]) {
      if (b->cls_count[c] == 0) continue;
      MHIP_CHECK(hipStreamWaitEvent(b->cs[c], b->ev[4], 0));
      launch_scf_class(b, b->cs[c], c, off, cap);
      MHIP_CHECK(hipEventRecord(b->ev[c], b->cs[c]));
    }
    if (b->bj && one_wg == 2)
      for (int it = 0; it < cap && one_iteration(b, true) > 0; ++it) {}
    for (int c = 0; c < one_wg; ++c)
      if (b->cls_count[c]) MHIP_CHECK(hipStreamWaitEvent(s, b->ev[c], 0));
    std::vector<BatchState> hs(b->nmol);
    MHIP_CHECK(hipMemcpyAsync(hs.data(), b->st.ptr, sizeof(BatchState) * b->nmol, hipMemcpyDeviceToHost, s));
    MHIP_CHECK(hipStreamSynchronize(s));
    const auto t1 = std::chrono::steady_clock::now();
    if (seconds) *seconds = std::chrono::duration<double>(t1 - t0).count();
    if (n_converged) {
      int c = 0;
      for (const auto& z : hs) c += converged(z) ? 1 : 0;
      *n_converged = c;
    }
  });
}

int mhip_batch_results(mhip_batch* b, double* escf, int* niter, int* conv) {
  return bguard([&] {
    std::vector<BatchState> hs(b->nmol);
    MHIP_CHECK(hipMemcpy(hs.data(), b->st.ptr, sizeof(BatchState) * b->nmol, hipMemcpyDeviceToHost));
    for (int m = 0; m < b->nmol; ++m) {
      if (escf) escf[m] = hs[m].escf;
      if (niter) niter[m] = hs[m].niter;
      if (conv) conv[m] = converged(hs[m]) ? 1 : 0;
    }
  });
}

int mhip_batch_density(mhip_batch* b, int m, double* p) {
  return bguard([&] {
    MHIP_REQUIRE(b && m >= 0 && m < b->nmol && p, "mhip_batch_density: bad arguments");
    long long off = 0;
    for (int k = 0; k < m; ++k) off += (long long)b->n_h[k] * (b->n_h[k] + 1) / 2;
    const long long mp = (long long)b->n_h[m] * (b->n_h[m] + 1) / 2;
    MHIP_CHECK(hipMemcpy(p, b->p.as<double>() + off, sizeof(double) * mp, hipMemcpyDeviceToHost));
  });
}

void mhip_batch_destroy(mhip_batch* b) {
  if (!b) return;
  (void)hipStreamSynchronize(b->s);
  bj_destroy(b->bj);
  for (auto c : b->cs)
    if (c) (void)hipStreamSynchronize(c), (void)hipStreamDestroy(c);
  for (auto e : b->ev)
    if (e) (void)hipEventDestroy(e);
  for (DevBuf* x : {&b->w, &b->h, &b->f, &b->p, &b->pa, &b->pold, &b->p1, &b->C, &b->global, &b->eig, &b->jrow,
                    &b->jcol, &b->nf0, &b->norb, &b->woff, &b->wcum, &b->w1off, &b->ccol, &b->heavy, &b->light,
                    &b->nhb, &b->nlb, &b->args, &b->mols, &b->cnv, &b->st, &b->act, &b->doeig, &b->mode, &b->niter,
                    &b->shift, &b->ee, &b->partial, &b->scal, &b->orboff, &b->atom_mol, &b->atom_idx,
                    &b->row_mol, &b->row_idx, &b->cls_list, &b->pdiag, &b->st0})
    x->release();
  (void)hipStreamDestroy(b->s);
  delete b;
}

}  // extern "C"
