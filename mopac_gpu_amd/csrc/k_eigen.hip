// FP64 symmetric eigensolver: parallel two-sided block Jacobi.
//
// The matrix (padded to a multiple of 64 with decoupled large diagonal
// entries) is split into 32-wide blocks.  A sweep visits every block pair once
// in round-robin order; a step turns every pair's two blocks by the orthogonal
// Q_pair that its 64x64 submatrix asks for (a workgroup per pair, in its LDS):
// A <- Qt^T A Qt tile by tile (two 64^3 products per tile), C <- C Qt.  One
// launch (k_jac_step) applies a step to A and C and solves the pairs of the
// next.  The comparison form (schedule 0: cyclic Jacobi over all 64 indices)
// takes three launches a step.
// In the SCF the solver starts from the previous eigenvectors (A = C^T F C is
// then nearly diagonal and one to three sweeps converge it); the first call
// starts from C = I.  Stopping test: max |A_ij| (i != j) <= tol * max|A_ii|.
#include <algorithm>
#include <cmath>

#include "common.h"
#include "k_eigen.h"
#include "k_jacobi_step.h"
#include "mfma.h"

namespace mhip {
namespace {

__device__ __forceinline__ void rr_pair(int round, int k, int& p, int& q) {
  // circle method on 64 indices: index 0 fixed, 1..63 rotate
  auto pos = [&](int slot) -> int { return slot == 0 ? 0 : 1 + ((slot - 1 + round) % 63); };
  p = pos(k);
  q = pos(63 - k);
}

constexpr int SOLVE_THREADS = 1024;

// Rotation k of round `round` from the current submatrix (cyclic Jacobi
// angle, the smaller of the two solutions).
__device__ __forceinline__ void pair_rotation(const double (*S)[LDSW], int round, int k, int& p, int& q,
                                              double& c, double& sn) {
  rr_pair(round, k, p, q);
  if (p > q) { const int t = p; p = q; q = t; }
  const double app = S[p][p], aqq = S[q][q], apq = S[p][q];
  c = 1.0;
  sn = 0.0;
  if (fabs(apq) > 1.0e-300 && fabs(apq) > 1.0e-18 * sqrt(fabs(app * aqq))) {
    // t = tan of the rotation angle, the root of t^2 + 2 theta t - 1 = 0
    // (theta = d / h) of smaller magnitude, written without theta:
    // t = sign(d) h / (|d| + sqrt(d^2 + h^2)); one division instead of three
    const double d = aqq - app, h = 2.0 * apq;
    double t = h / (fabs(d) + sqrt(d * d + h * h));
    if (d < 0.0) t = -t;
    c = rsqrt(t * t + 1.0);
    sn = t * c;
  }
}

// One workgroup per block pair: load the 64x64 submatrix, run cyclic Jacobi
// in parallel (round-robin) order until converged or max_inner sweeps, and
// write the accumulated rotation Q.  A pair already diagonal to `skip_abs`
// is marked inactive (Q = I) and skipped by the update kernels.
//
// A round: the first wave computes the round's 32 disjoint rotations into
// LDS; then the 1024 threads each own one 2x2 block (row pair k1, column pair
// k2) of the submatrix and apply rotation k1 to its rows and k2 to its
// columns in one pass, in place (no other thread touches the block), and
// rotate two rows of Q's columns p(k2), q(k2).  Two barriers per round.
__global__ __launch_bounds__(SOLVE_THREADS) void k_jac_solve(
    const double* __restrict__ A, int lda, int nreal, const int* __restrict__ pairs,
    double* __restrict__ Qbuf, int* __restrict__ active, double tol, double skip_abs,
    int max_inner) {
  static_assert(SOLVE_THREADS == (SB / 2) * (SB / 2), "one thread per 2x2 block");
  __shared__ double S[SB][LDSW];
  __shared__ double Q[SB][LDSW];
  __shared__ double rc[32], rs[32];
  __shared__ int rp[32], rq[32];
  __shared__ double red_off[SOLVE_THREADS / 64], red_dg[SOLVE_THREADS / 64];
  const int pidx = blockIdx.x;
  const int I = pairs[2 * pidx], J = pairs[2 * pidx + 1];
  const int tid = threadIdx.x;
  const int k1 = tid >> 5, k2 = tid & 31;
  {
    // all four loads of this thread in flight before the first LDS store
    constexpr int PER = SB * SB / SOLVE_THREADS;
    double v[PER];
#pragma unroll
    for (int it = 0; it < PER; ++it) {
      const int e = tid + SOLVE_THREADS * it;
      v[it] = A[(size_t)gidx_dev(I, J, e % SB) + (size_t)gidx_dev(I, J, e / SB) * lda];
    }
#pragma unroll
    for (int it = 0; it < PER; ++it) {
      const int e = tid + SOLVE_THREADS * it, r = e % SB, c = e / SB;
      S[r][c] = v[it];
      Q[r][c] = (r == c) ? 1.0 : 0.0;
    }
  }
  __syncthreads();
  for (int sw = 0; sw < max_inner; ++sw) {
    double off = 0.0, dg = 0.0;
    for (int e = tid; e < SB * SB; e += SOLVE_THREADS) {
      const int r = e % SB, c = e / SB;
      if (r == c) {
        if (gidx_dev(I, J, r) < nreal) dg = fmax(dg, fabs(S[r][c]));
      } else {
        off = fmax(off, fabs(S[r][c]));
      }
    }
    off = wave_max(off);
    dg = wave_max(dg);
    if ((tid & 63) == 0) {
      red_off[tid >> 6] = off;
      red_dg[tid >> 6] = dg;
    }
    __syncthreads();
    off = 0.0;
    dg = 0.0;
#pragma unroll
    for (int w = 0; w < SOLVE_THREADS / 64; ++w) {
      off = fmax(off, red_off[w]);
      dg = fmax(dg, red_dg[w]);
    }
    __syncthreads();
    if (sw == 0 && off <= skip_abs) {
      if (tid == 0) active[pidx] = 0;
      return;
    }
    if (off <= tol * fmax(dg, 1.0)) break;
    for (int round = 0; round < 63; ++round) {
      if (tid < 32) {
        int p, q;
        double c, sn;
        pair_rotation(S, round, tid, p, q, c, sn);
        rc[tid] = c; rs[tid] = sn; rp[tid] = p; rq[tid] = q;
      }
      __syncthreads();
      const int p1 = rp[k1], q1 = rq[k1], p2 = rp[k2], q2 = rq[k2];
      const double c1 = rc[k1], s1 = rs[k1], c2 = rc[k2], s2 = rs[k2];
      const double xpp = S[p1][p2], xpq = S[p1][q2], xqp = S[q1][p2], xqq = S[q1][q2];
      // rows p1, q1 (rotation k1), then columns p2, q2 (rotation k2)
      const double rpp = c1 * xpp - s1 * xqp, rpq = c1 * xpq - s1 * xqq;
      const double rqp = s1 * xpp + c1 * xqp, rqq = s1 * xpq + c1 * xqq;
      S[p1][p2] = c2 * rpp - s2 * rpq;
      S[p1][q2] = s2 * rpp + c2 * rpq;
      S[q1][p2] = c2 * rqp - s2 * rqq;
      S[q1][q2] = s2 * rqp + c2 * rqq;
      // Q <- Q J(k2) on rows 2 k1, 2 k1 + 1
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int row = 2 * k1 + h;
        const double u = Q[row][p2], v = Q[row][q2];
        Q[row][p2] = c2 * u - s2 * v;
        Q[row][q2] = s2 * u + c2 * v;
      }
      __syncthreads();
    }
  }
  double* Qo = Qbuf + (size_t)pidx * SB * SB;
  for (int e = tid; e < SB * SB; e += SOLVE_THREADS) {
    const int r = e % SB, c = e / SB;
    Qo[e] = Q[r][c];
  }
  if (tid == 0) active[pidx] = 1;
}

__global__ __launch_bounds__(CROSS_THREADS, 4) void k_jac_solve_x(
    const double* __restrict__ A, int lda, int nreal, const int* __restrict__ pairs,
    const int* __restrict__ intra, double* __restrict__ Qbuf, int* __restrict__ active, double* __restrict__ diag,
    double tol, double skip_abs, int max_inner, SweepTest test) {
  __shared__ JacLds lds;
  if (test.done(skip_abs)) return;
  const int pidx = blockIdx.x;
  const int I = pairs[2 * pidx], J = pairs[2 * pidx + 1];
  solve_from_memory(lds, A, lda, I, J, intra[pidx] != 0,
                    JacSolve{nreal, Qbuf + (size_t)pidx * SB * SB, active + pidx,
                             diag ? diag + (size_t)I * BS * BS : nullptr, diag ? diag + (size_t)J * BS * BS : nullptr,
                             tol, skip_abs, max_inner});
}

// A(rows of pair P1, cols of pair P2) <- Q1^T A Q2 for P1 <= P2 (the mirror
// tile is written as the transpose, keeping A exactly symmetric).
__global__ __launch_bounds__(256) void k_jac_apply_a(double* __restrict__ A, int lda, int npairs,
                                                     int npo, const int* __restrict__ pairs,
                                                     const double* __restrict__ Qbuf,
                                                     const int* __restrict__ active) {
  // blockIdx.x enumerates (P1 <= P2)
  int P1, P2;
  tile_of(blockIdx.x, npairs, npo, P1, P2);
  const bool a1 = active[P1] != 0, a2 = active[P2] != 0;
  if (!a1 && !a2) return;
  __shared__ double At[SB][LDSW];
  __shared__ double Q1[SB][LDSW];
  __shared__ double Q2[SB][LDSW];
  const int I1 = pairs[2 * P1], J1 = pairs[2 * P1 + 1];
  const int I2 = pairs[2 * P2], J2 = pairs[2 * P2 + 1];
  const int tid = threadIdx.x;
  const double* q1 = Qbuf + (size_t)P1 * SB * SB;
  const double* q2 = Qbuf + (size_t)P2 * SB * SB;
  for (int e = tid; e < SB * SB; e += 256) {
    const int r = e % SB, c = e / SB;
    At[r][c] = A[(size_t)gidx(I1, J1, r) + (size_t)gidx(I2, J2, c) * lda];
    Q1[r][c] = a1 ? q1[e] : (r == c ? 1.0 : 0.0);
    Q2[r][c] = a2 ? q2[e] : (r == c ? 1.0 : 0.0);
  }
  __syncthreads();
  const int tx = tid & 15, ty = tid >> 4;
  double acc[4][4] = {};
  // T = Q1^T At : T[r][c] = sum_k Q1[k][r] At[k][c]
  for (int k = 0; k < SB; ++k) {
    double a4[4], b4[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) a4[i] = Q1[k][ty * 4 + i];
#pragma unroll
    for (int j = 0; j < 4; ++j) b4[j] = At[k][tx * 4 + j];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = fma(a4[i], b4[j], acc[i][j]);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) At[ty * 4 + i][tx * 4 + j] = acc[i][j];
  __syncthreads();
  double out[4][4] = {};
  // Out = T Q2 : Out[r][c] = sum_k T[r][k] Q2[k][c]
  for (int k = 0; k < SB; ++k) {
    double a4[4], b4[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) a4[i] = At[ty * 4 + i][k];
#pragma unroll
    for (int j = 0; j < 4; ++j) b4[j] = Q2[k][tx * 4 + j];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) out[i][j] = fma(a4[i], b4[j], out[i][j]);
  }
  if (P1 == P2) {
    // diagonal tile: symmetrize exactly
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) At[ty * 4 + i][tx * 4 + j] = out[i][j];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = ty * 4 + i, c = tx * 4 + j;
        const double v = (r == c) ? out[i][j] : 0.5 * (out[i][j] + At[c][r]);
        A[(size_t)gidx(I1, J1, r) + (size_t)gidx(I2, J2, c) * lda] = v;
      }
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = ty * 4 + i, c = tx * 4 + j;
      const size_t gr = gidx(I1, J1, r), gc = gidx(I2, J2, c);
      A[gr + gc * lda] = out[i][j];
      A[gc + gr * lda] = out[i][j];
    }
}

// C(rows tile, cols of pair P) <- C(rows tile, cols of P) Q_P
__global__ __launch_bounds__(256) void k_jac_apply_c(double* __restrict__ C, int ldc, int nrows,
                                                     const int* __restrict__ pairs,
                                                     const double* __restrict__ Qbuf,
                                                     const int* __restrict__ active) {
  const int P = blockIdx.y;
  if (!active[P]) return;
  __shared__ double Ct[SB][LDSW];
  __shared__ double Qs[SB][LDSW];
  const int row0 = blockIdx.x * SB;
  const int I = pairs[2 * P], J = pairs[2 * P + 1];
  const double* q = Qbuf + (size_t)P * SB * SB;
  const int tid = threadIdx.x;
  for (int e = tid; e < SB * SB; e += 256) {
    const int r = e % SB, c = e / SB;
    const int gr = row0 + r;
    Ct[r][c] = (gr < nrows) ? C[(size_t)gr + (size_t)gidx(I, J, c) * ldc] : 0.0;
    Qs[r][c] = q[e];
  }
  __syncthreads();
  const int tx = tid & 15, ty = tid >> 4;
  double out[4][4] = {};
  for (int k = 0; k < SB; ++k) {
    double a4[4], b4[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) a4[i] = Ct[ty * 4 + i][k];
#pragma unroll
    for (int j = 0; j < 4; ++j) b4[j] = Qs[k][tx * 4 + j];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) out[i][j] = fma(a4[i], b4[j], out[i][j]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int gr = row0 + ty * 4 + i;
    if (gr >= nrows) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) C[(size_t)gr + (size_t)gidx(I, J, tx * 4 + j) * ldc] = out[i][j];
  }
}


// Workgroups [0, npairs) solve the next step's pairs, the next ntiles update
// A, the others C.  The solves are the longest and start first; they read A
// before the step while the update writes the other buffer, so nothing in
// the launch waits for anything else in it.
//
// Solving in a launch of its own left the chip to npairs workgroups for 22
// of a step's 37 us at 1020 orbitals (with the A update behind it, and the C
// update on a second stream, ordered by two events per step); this launch
// takes 22 us, of which the solve's 32 rounds are 12 and putting its problem
// together 4.  At 3072 orbitals the updates set it: 54 us, 40 in two groups.
__global__ __launch_bounds__(CROSS_THREADS, 4) void k_jac_step(JacStep a, int base, SweepTest test) {
  static_assert(UPD_NT == CROSS_THREADS, "one workgroup size for every role");
  __shared__ JacLds lds;
  if (test.done(a.skip_abs)) return;
  const int b = (int)blockIdx.x + base;
  if (b < a.npairs) {
    step_solve(lds, a, b);
  } else if (b < a.npairs + a.ntiles) {
    step_tile_a(lds.m, a, b - a.npairs);
  } else {
    // tiles of C; of two diagonal blocks only theirs
    const int c = b - a.npairs - a.ntiles, nrow = a.lda / SB, rows0 = a.crows ? a.crows : nrow, n0 = a.npo * rows0;
    if (c < n0) step_tile_c(lds.m, a, (c % rows0) * SB, c / rows0);
    else step_tile_c(lds.m, a, (rows0 + (c - n0) % (nrow - rows0)) * SB, a.npo + (c - n0) / (nrow - rows0));
  }
}

// max |A_ij| (i != j) and max |A_ii| over the leading n x n block.
// split > 0: only entries inside [0, split) x [0, split) and its complement
// count (the grouped schedule never rotates across the two groups)
__global__ __launch_bounds__(256) void k_offmax_partial(int n, const double* __restrict__ A,
                                                        int lda, int split, double* __restrict__ part) {
  const int j = blockIdx.x;
  double off = 0.0, dg = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) {
    const double v = fabs(A[(size_t)i + (size_t)j * lda]);
    if (i == j) dg = v;
    else if (split <= 0 || ((i < split) == (j < split))) off = fmax(off, v);
  }
  __shared__ double r1[256], r2[256];
  r1[threadIdx.x] = off;
  r2[threadIdx.x] = dg;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) {
      r1[threadIdx.x] = fmax(r1[threadIdx.x], r1[threadIdx.x + w]);
      r2[threadIdx.x] = fmax(r2[threadIdx.x], r2[threadIdx.x + w]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * j] = r1[0];
    part[2 * j + 1] = r2[0];
  }
}

__global__ __launch_bounds__(1024) void k_offmax_final(int n, const double* __restrict__ part,
                                                       double* __restrict__ out, double* __restrict__ host) {
  double off = 0.0, dg = 0.0;
  for (int j = threadIdx.x; j < n; j += 1024) {
    off = fmax(off, part[2 * j]);
    dg = fmax(dg, part[2 * j + 1]);
  }
  __shared__ double r1[1024], r2[1024];
  r1[threadIdx.x] = off;
  r2[threadIdx.x] = dg;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if (threadIdx.x < w) {
      r1[threadIdx.x] = fmax(r1[threadIdx.x], r1[threadIdx.x + w]);
      r2[threadIdx.x] = fmax(r2[threadIdx.x], r2[threadIdx.x + w]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = host[0] = r1[0];
    out[1] = host[1] = r2[0];
  }
}

// A by 2^e
__global__ __launch_bounds__(256) void k_scale_by_power(long long len, double* __restrict__ A, int e) {
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < len; i += (long long)gridDim.x * 256)
    A[i] = ldexp(A[i], e);
}

// active pairs of the step in each group: out[0] over [0, npo), out[1] over [npo, npairs)
__global__ void k_count_active(int npairs, int npo, const int* __restrict__ active, int* __restrict__ out) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    int a = 0, b = 0;
    for (int i = 0; i < npairs; ++i) {
      if (i < npo) a += active[i] != 0;
      else b += active[i] != 0;
    }
    out[0] = a;
    out[1] = b;
  }
}

// Stable ascending rank sort of the diagonal; perm[rank] = index.  64 entries
// per workgroup, a wave for every eighth of the others; the diagonal goes
// through LDS in chunks.  A thread per entry compared with all of them, in
// four workgroups at 1020 orbitals, took 74 us; this takes 12.
constexpr int SORT_CHUNK = 2048, SORT_WAVES = 8;
__global__ __launch_bounds__(64 * SORT_WAVES) void k_sort_diag(int n, int npad, const double* __restrict__ A, int lda,
                                                               int* __restrict__ perm, double* __restrict__ eig) {
  __shared__ double d[SORT_CHUNK];
  __shared__ int below[SORT_WAVES][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = blockIdx.x * 64 + lane;
  const double level = (i < npad) ? A[(size_t)i + (size_t)i * lda] : 0.0, di = sort_key(level, i, n);
  int rank = 0;
  for (int j0 = 0; j0 < npad; j0 += SORT_CHUNK) {
    const int nj = min(SORT_CHUNK, npad - j0);
    for (int j = threadIdx.x; j < nj; j += 64 * SORT_WAVES)
      d[j] = sort_key(A[(size_t)(j0 + j) + (size_t)(j0 + j) * lda], j0 + j, n);
    __syncthreads();
#pragma unroll 8
    for (int j = w; j < nj; j += SORT_WAVES) {
      const double dj = d[j];
      rank += (dj < di) || (dj == di && j0 + j < i);
    }
    __syncthreads();
  }
  below[w][lane] = rank;
  __syncthreads();
  if (w == 0 && i < npad) {
    for (int v = 1; v < SORT_WAVES; ++v) rank += below[v][lane];
    perm[rank] = i;
    eig[rank] = level;
  }
}

__global__ void k_permute_cols(int nrows, int ncols, const double* __restrict__ src, int lds,
                               const int* __restrict__ perm, double* __restrict__ dst, int ldd) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = blockIdx.y;
  if (r >= nrows || k >= ncols) return;
  dst[(size_t)r + (size_t)k * ldd] = src[(size_t)r + (size_t)perm[k] * lds];
}

__global__ void k_set_identity(int npad, double* __restrict__ C, int ldc) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  const int c = blockIdx.y;
  if (r >= npad) return;
  C[(size_t)r + (size_t)c * ldc] = (r == c) ? 1.0 : 0.0;
}

// Largest-|c| coefficient of each column made positive (first occurrence wins).
__global__ __launch_bounds__(256) void k_phase_lock(int n, double* __restrict__ C, int ldc) {
  const int col = blockIdx.x;
  double* v = C + (size_t)col * ldc;
  double best = 0.0, sgn = 0.0;
  int bi = n;
  for (int r = threadIdx.x; r < n; r += 256) {
    const double a = fabs(v[r]);
    if (a > best) { best = a; sgn = v[r]; bi = r; }
  }
  __shared__ double sb[256], ss[256];
  __shared__ int si[256];
  sb[threadIdx.x] = best; ss[threadIdx.x] = sgn; si[threadIdx.x] = bi;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) {
      const double b2 = sb[threadIdx.x + w];
      const int i2 = si[threadIdx.x + w];
      if (b2 > sb[threadIdx.x] || (b2 == sb[threadIdx.x] && i2 < si[threadIdx.x])) {
        sb[threadIdx.x] = b2; ss[threadIdx.x] = ss[threadIdx.x + w]; si[threadIdx.x] = i2;
      }
    }
    __syncthreads();
  }
  const bool flip = ss[0] < 0.0;
  if (flip)
    for (int r = threadIdx.x; r < n; r += 256) v[r] = -v[r];
}

}  // namespace

int g_jacobi_schedule = 1;

void JacobiPlan::build(int n_in, int split) {
  n = n_in;
  npad = ((n + SB - 1) / SB) * SB;
  nb = npad / BS;
  npairs = nb / 2;
  // circle method over the blocks [b0, b0 + m): round r, pair k
  auto circle = [](int b0, int m, int r, int k, int& a, int& b) {
    auto pos = [&](int slot) { return slot == 0 ? 0 : 1 + ((slot - 1 + r) % (m - 1)); };
    a = b0 + pos(k);
    b = b0 + pos(m - 1 - k);
    if (a > b) std::swap(a, b);
  };
  const int nbo = (split > 0 && split % BS == 0) ? split / BS : 0;
  const int nbv = nb - nbo;
  grouped = nbo >= 2 && nbv >= 2 && nbo % 2 == 0 && nbv % 2 == 0;
  this->split = grouped ? split : 0;
  npo = grouped ? nbo / 2 : npairs;
  std::vector<int> h;
  if (grouped) {
    // two independent problems (blocks [0, nbo) and [nbo, nb)) in every
    // step; the smaller one repeats its rounds while the larger finishes
    nsteps = std::max(nbo, nbv) - 1;
    h.resize((size_t)nsteps * npairs * 2);
    for (int step = 0; step < nsteps; ++step) {
      int k = 0;
      for (int q = 0; q < nbo / 2; ++q, ++k)
        circle(0, nbo, step % (nbo - 1), q, h[((size_t)step * npairs + k) * 2],
               h[((size_t)step * npairs + k) * 2 + 1]);
      for (int q = 0; q < nbv / 2; ++q, ++k)
        circle(nbo, nbv, step % (nbv - 1), q, h[((size_t)step * npairs + k) * 2],
               h[((size_t)step * npairs + k) * 2 + 1]);
    }
  } else {
    nsteps = nb - 1;
    h.resize((size_t)nsteps * npairs * 2);
    for (int step = 0; step < nsteps; ++step)
      for (int k = 0; k < npairs; ++k)
        circle(0, nb, step, k, h[((size_t)step * npairs + k) * 2], h[((size_t)step * npairs + k) * 2 + 1]);
  }
  pairs.ensure(h.size() * sizeof(int));
  MHIP_CHECK(hipMemcpy(pairs.ptr, h.data(), h.size() * sizeof(int), hipMemcpyHostToDevice));
  // intra-block rounds at the first step of each sweep of a pair's group
  std::vector<int> fl((size_t)nsteps * npairs, 0);
  for (int step = 0; step < nsteps; ++step)
    for (int k = 0; k < npairs; ++k) {
      const bool first = grouped ? (k < npo ? step % (nbo - 1) == 0 : step % (nbv - 1) == 0) : step == 0;
      fl[(size_t)step * npairs + k] = first ? 1 : 0;
    }
  intra_host = fl;
  intra.ensure(fl.size() * sizeof(int));
  MHIP_CHECK(hipMemcpy(intra.ptr, fl.data(), fl.size() * sizeof(int), hipMemcpyHostToDevice));
  // where each block is in each step
  std::vector<int> wh((size_t)nsteps * nb, 0);
  for (int step = 0; step < nsteps; ++step)
    for (int k = 0; k < npairs; ++k)
      for (int half = 0; half < 2; ++half)
        wh[(size_t)step * nb + h[((size_t)step * npairs + k) * 2 + half]] = 2 * k + half;
  where.ensure(wh.size() * sizeof(int));
  MHIP_CHECK(hipMemcpy(where.ptr, wh.data(), wh.size() * sizeof(int), hipMemcpyHostToDevice));
  // rotations, flags and diagonal blocks of two consecutive steps
  qbuf.ensure((size_t)2 * npairs * SB * SB * sizeof(double));
  diag.ensure((size_t)2 * nb * BS * BS * sizeof(double));
  active.ensure((size_t)2 * npairs * sizeof(int));
  part.ensure((size_t)2 * npad * sizeof(double) + 64);
  perm.ensure((size_t)npad * sizeof(int));
  counts.ensure((size_t)2 * nsteps * sizeof(int));
}

void JacobiPlan::ensure_test_event(hipStream_t s) {
  if (tested) return;
  // an event belongs to the device that is current, a stream to its own
  int device = 0, of_stream = 0;
  MHIP_CHECK(hipGetDevice(&device));
  MHIP_CHECK(hipStreamGetDevice(s, &of_stream));
  if (device != of_stream) MHIP_CHECK(hipSetDevice(of_stream));
  const hipError_t r = hipEventCreateWithFlags(&tested, hipEventDisableTiming);
  if (device != of_stream) (void)hipSetDevice(device);
  MHIP_CHECK(r);
}

void jacobi_set_identity(hipStream_t s, int npad, double* C, int ldc) {
  hipLaunchKernelGGL(k_set_identity, dim3((npad + 255) / 256, npad), dim3(256), 0, s, npad, C, ldc);
  MHIP_LAUNCH_CHECK();
}

// jacobi_sweeps on a matrix whose elements end at kAngleRange in the cross
// schedule; one with larger ones is left alone, and returns 2 with the test's
// two values in host_scal.
static int sweeps_in_range(hipStream_t s, JacobiPlan& plan, double*& A, double*& A2, double* C, double tol,
                           int max_sweeps, double* host_scal, double* dev_scal, int* sweeps_done, bool c_blocks) {
  const int lda = plan.npad;
  int done = 0;
  // Inner sweeps per step.  Cross schedule: one; a second saves up to a fifth
  // of the sweeps (54 instead of 66 in the plain SCF of 1020 orbitals) for
  // twice the rounds (72 ms instead of 58; 12.1 instead of 9.7 ms at 174
  // orbitals).  A matrix that is one pair problem is solved in one launch.
  const bool cross = g_jacobi_schedule == 1;
  const int inner = plan.max_inner > 0 ? plan.max_inner : !cross ? 2 : plan.npairs == 1 ? 16 : 1;
  const double inner_tol = plan.npairs == 1 ? 0.5 * tol : 1.0e-14;
  // every step's solves ride in the launch of the step before
  const bool ahead = cross && g_kernel_variant == 1 && plan.npairs > 1;
  const int npairs = plan.npairs, npv = npairs - plan.npo, nsteps = plan.nsteps;
  const int ntiles = plan.npo * (plan.npo + 1) / 2 + npv * (npv + 1) / 2, nrow = plan.npad / SB;
  const int crows = c_blocks ? plan.split / SB : 0;
  const int nctiles = crows ? plan.npo * crows + npv * (nrow - crows) : npairs * nrow;
  int slot = 0;  // of the step at hand in the two-step buffers
  auto qslot = [&](int k) { return plan.qbuf.as<double>() + (size_t)k * npairs * SB * SB; };
  auto aslot = [&](int k) { return plan.active.as<int>() + (size_t)k * npairs; };
  auto dslot = [&](int k) { return plan.diag.as<double>() + (size_t)k * plan.nb * BS * BS; };
  auto pairs_of = [&](int step) { return plan.pairs.as<int>() + (size_t)step * npairs * 2; };
  auto intra_of = [&](int step) { return plan.intra.as<int>() + (size_t)step * npairs; };
  auto solve = [&](int step, double skip_abs, SweepTest test = {}) {
    if (cross)
      hipLaunchKernelGGL(k_jac_solve_x, dim3(npairs), dim3(CROSS_THREADS), 0, s, A, lda, plan.n, pairs_of(step),
                         intra_of(step), qslot(slot), aslot(slot), ahead ? dslot(slot) : nullptr, inner_tol, skip_abs,
                         inner, test);
    else
      hipLaunchKernelGGL(k_jac_solve, dim3(npairs), dim3(SOLVE_THREADS), 0, s, A, lda, plan.n, pairs_of(step),
                         qslot(slot), aslot(slot), 1.0e-14, skip_abs, inner);
    MHIP_LAUNCH_CHECK();
  };
  // A solve shares its CU with an update workgroup where two fit, and takes
  // longer for it.  While the updates need no more than about three rounds of
  // the chip one to a CU, they still end before the solves: LDS that is not
  // used keeps every workgroup alone.  SCFs at 1020 orbitals (408 workgroups)
  // 53.3 -> 49.4 ms, 1200 (570) 71.2 -> 66.4, 1500 (900) equal, 1800 (1305)
  // 133 -> 160.
  const int total = npairs + ntiles + nctiles;
  const size_t alone = total <= 3 * 256 ? 16384 : 0;
  auto launch_step = [&](int step, double skip_abs, int from, int to, SweepTest test) {
    const int next = (step + 1) % nsteps;
    const JacStep a{A,          ahead ? A2 : A,  C,                lda,
                    plan.n,     npairs,          plan.npo,         ntiles,
                    pairs_of(step), qslot(slot), aslot(slot),      pairs_of(next),
                    intra_of(next), plan.where.as<int>() + (size_t)step * plan.nb, qslot(slot ^ 1), aslot(slot ^ 1),
                    dslot(slot), dslot(slot ^ 1), inner_tol,       skip_abs,
                    inner,      crows};
    auto launch = [&] {
      hipLaunchKernelGGL(k_jac_step, dim3(to - from), dim3(CROSS_THREADS), alone, s, a, from, test);
      MHIP_LAUNCH_CHECK();
    };
    if (ahead && to - from == total) timed(s, K_JACOBI, 0.0, 0.0, launch);
    else launch();
  };
  plan.ensure_test_event(s);
  for (int sw = 0; sw <= max_sweeps; ++sw) {
    hipLaunchKernelGGL(k_offmax_partial, dim3(plan.n), dim3(256), 0, s, plan.n, A, lda,
                       plan.grouped ? plan.split : 0, plan.part.as<double>());
    MHIP_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_offmax_final, dim3(1), dim3(1024), 0, s, plan.n, plan.part.as<double>(), dev_scal,
                       host_scal);
    MHIP_LAUNCH_CHECK();
    MHIP_CHECK(hipEventRecord(plan.tested, s));
    const bool timing = plan.timing && g_kernel_variant == 1;
    // The sweep's first launch waits on the device for the test's outcome, not
    // for the host's: it runs while the host learns it, or does nothing.
    const bool early = ahead && !timing && sw < max_sweeps;
    if (early) {
      const SweepTest test{dev_scal, tol, sw == 0};
      if (sw == 0) solve(0, 0.0, test);
      else launch_step(0, 0.0, 0, total, test);
    }
    MHIP_CHECK(hipEventSynchronize(plan.tested));
    const double thr = tol * std::max(1.0, host_scal[1]);
    if (host_scal[0] <= thr) break;
    const double top = std::max(host_scal[0], host_scal[1]);
    if (cross && sw == 0 && top > kAngleRange && std::isfinite(top)) return 2;
    // pairs whose whole 64x64 block is already this diagonal are left alone
    const double skip_abs = 0.1 * thr;
    if (sw == max_sweeps) {
      if (sweeps_done) *sweeps_done = done;
      return 1;
    }
    if (plan.timing && plan.ev.size() < (size_t)(6 * nsteps)) {
      for (auto e : plan.ev) (void)hipEventDestroy(e);
      plan.ev.assign(6 * nsteps, nullptr);
      for (auto& e : plan.ev) MHIP_CHECK(hipEventCreate(&e));
    }
    // part k of the step's launch between events 2 k and 2 k + 1
    auto mark = [&](int step, int k) {
      if (timing) MHIP_CHECK(hipEventRecord(plan.ev[6 * step + k], s));
    };
    // the first step's solve of a later sweep ran in the last launch of the
    // sweep before
    if (ahead && sw == 0 && !early) solve(0, skip_abs);
    for (int step = 0; step < nsteps; ++step) {
      if (!ahead) {
        mark(step, 0);
        solve(step, skip_abs);
        mark(step, 1);
      }
      if (timing)
        hipLaunchKernelGGL(k_count_active, dim3(1), dim3(64), 0, s, npairs, plan.npo, aslot(slot),
                           plan.counts.as<int>() + 2 * step);
      if (g_kernel_variant == 1) {
        if (!timing) {
          if (!early || sw == 0 || step > 0) launch_step(step, skip_abs, ahead ? 0 : npairs, total, {});
        } else {
          // the same work in a launch per part, for the parts' times
          if (ahead) {
            mark(step, 0);
            launch_step(step, skip_abs, 0, npairs, {});
            mark(step, 1);
          }
          mark(step, 2);
          launch_step(step, skip_abs, npairs, npairs + ntiles, {});
          mark(step, 3);
          mark(step, 4);
          launch_step(step, skip_abs, npairs + ntiles, total, {});
          mark(step, 5);
        }
        if (ahead) {
          std::swap(A, A2);
          slot ^= 1;
        }
      } else {
        hipLaunchKernelGGL(k_jac_apply_a, dim3(ntiles), dim3(256), 0, s, A, lda, npairs, plan.npo, pairs_of(step),
                           qslot(slot), aslot(slot));
        MHIP_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_jac_apply_c, dim3(plan.npad / SB, npairs), dim3(256), 0, s, C, lda, plan.npad,
                           pairs_of(step), qslot(slot), aslot(slot));
        MHIP_LAUNCH_CHECK();
      }
    }
    if (timing) {
      MHIP_CHECK(hipStreamSynchronize(s));
      std::vector<int> act(2 * nsteps);
      MHIP_CHECK(hipMemcpy(act.data(), plan.counts.ptr, sizeof(int) * 2 * nsteps, hipMemcpyDeviceToHost));
      for (int step = 0; step < nsteps; ++step) {
        // tiles processed: those of each group with at least one active pair
        const long long u0 = plan.npo - act[2 * step], u1 = npv - act[2 * step + 1];
        plan.active_pairs += act[2 * step] + act[2 * step + 1];
        // a full inner sweep is 2016 rotations; cross rounds are 32 x 32,
        // plus 2 x 496 inside the blocks where the step's intra flag is set
        for (int g = 0; g < 2; ++g) {
          const int first = g == 0 ? 0 : plan.npo;
          if (first >= npairs) continue;
          const long long per =
              cross ? 1024 + (plan.intra_host[(size_t)step * npairs + first] ? 992 : 0) : 2016LL * inner;
          plan.active_rotations += per * act[2 * step + g];
        }
        plan.active_tiles += (long long)ntiles - u0 * (u0 + 1) / 2 - u1 * (u1 + 1) / 2;
        float t[3];
        for (int k = 0; k < 3; ++k)
          MHIP_CHECK(hipEventElapsedTime(&t[k], plan.ev[6 * step + 2 * k], plan.ev[6 * step + 2 * k + 1]));
        plan.t_solve_ms += t[0];
        plan.t_apply_ms += t[1];
        plan.t_applyc_ms += t[2];
        plan.n_solve++;
        plan.n_apply++;
        plan.n_applyc++;
      }
    }
    ++done;
  }
  if (sweeps_done) *sweeps_done = done;
  return 0;
}

int jacobi_sweeps(hipStream_t s, JacobiPlan& plan, double*& A, double*& A2, double* C, double tol, int max_sweeps,
                  double* host_scal, double* dev_scal, int* sweeps_done, bool c_blocks) {
  int rc = sweeps_in_range(s, plan, A, A2, C, tol, max_sweeps, host_scal, dev_scal, sweeps_done, c_blocks);
  if (rc != 2) return rc;
  // the largest element to 2^10, above the 1 that the stopping test takes for
  // the diagonal of a smaller one
  const int e = std::ilogb(std::max(host_scal[0], host_scal[1])) - 10;
  const long long len = (long long)plan.npad * plan.npad;
  auto scale = [&](int by) {
    hipLaunchKernelGGL(k_scale_by_power, dim3((int)std::min<long long>(4096, (len + 255) / 256)), dim3(256), 0, s, len,
                       A, by);
    MHIP_LAUNCH_CHECK();
  };
  scale(-e);
  rc = sweeps_in_range(s, plan, A, A2, C, tol, max_sweeps, host_scal, dev_scal, sweeps_done, c_blocks);
  scale(e);
  return rc;
}

void jacobi_sort(hipStream_t s, JacobiPlan& plan, const double* A, const double* C, double* Cout,
                 double* eig_dev) {
  const int npad = plan.npad;
  hipLaunchKernelGGL(k_sort_diag, dim3((npad + 63) / 64), dim3(64 * SORT_WAVES), 0, s, plan.n, npad, A, npad,
                     plan.perm.as<int>(), eig_dev);
  MHIP_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_permute_cols, dim3((npad + 255) / 256, npad), dim3(256), 0, s, npad, npad, C,
                     npad, plan.perm.as<int>(), Cout, npad);
  MHIP_LAUNCH_CHECK();
}

void phase_lock(hipStream_t s, int n, double* C, int ldc) {
  hipLaunchKernelGGL(k_phase_lock, dim3(n), dim3(256), 0, s, n, C, ldc);
  MHIP_LAUNCH_CHECK();
}

}  // namespace mhip
