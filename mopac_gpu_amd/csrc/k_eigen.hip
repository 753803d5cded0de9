// FP64 symmetric eigensolver: parallel two-sided block Jacobi.
//
// The matrix (padded to a multiple of 64 with decoupled large diagonal
// entries) is split into 32-wide blocks.  A sweep visits every block pair once
// in round-robin order; each step
//   1. diagonalizes the 64x64 submatrix of every pair in LDS (inner cyclic
//      Jacobi, one workgroup per pair) giving an orthogonal Q_pair,
//   2. applies A <- Qt^T A Qt tile by tile (two 64^3 products per tile),
//   3. applies C <- C Qt to the eigenvector accumulator.
// In the SCF the solver starts from the previous eigenvectors (A = C^T F C is
// then nearly diagonal and one to three sweeps converge it); the first call
// starts from C = I.  Stopping test: max |A_ij| (i != j) <= tol * max|A_ii|.
#include <utility>

#include "common.h"
#include "k_eigen.h"
#include "mfma.h"

namespace mhip {
namespace {

constexpr int BS = 32;  // block width
constexpr int SB = 64;  // pair width
constexpr int LDSW = SB + 1;

__device__ __forceinline__ int gidx_dev(int pairI, int pairJ, int local) {
  return (local < BS) ? pairI * BS + local : pairJ * BS + (local - BS);
}

__device__ __forceinline__ void rr_pair(int round, int k, int& p, int& q) {
  // circle method on 64 indices: index 0 fixed, 1..63 rotate
  auto pos = [&](int slot) -> int { return slot == 0 ? 0 : 1 + ((slot - 1 + round) % 63); };
  p = pos(k);
  q = pos(63 - k);
}

constexpr int SOLVE_THREADS = 1024;

__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}

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

// Angle of the rotation that zeroes apq in [[app, apq], [apq, aqq]], the
// root t of h t^2 + 2 d t - h = 0 (d = aqq - app, h = 2 apq) of smaller
// magnitude: after it the diagonal is app - t apq, aqq + t apq.  The root
// comes from FP32 (reciprocal and square root in one instruction each) and
// one FP64 Newton step, which leaves it good to about 1e-13; what an angle
// error leaves of apq goes to the next sweep.  c = 1 / sqrt(1 + t^2) is
// refined to the last bit in FP64, so c^2 + s^2 = 1 as for the exact angle.
// About 25 dependent operations instead of the 100 of an FP64 division and
// two square roots.
__device__ __forceinline__ void rotation_of(double app, double aqq, double apq, double& c, double& sn,
                                            double& t) {
  c = 1.0;
  sn = 0.0;
  t = 0.0;
  const double d = aqq - app, h = 2.0 * apq;
  const float df = (float)d, hf = (float)h;
  // |apq| > 1e-18 sqrt|app aqq| compared as squares; below FP32's range an
  // element is left as it is
  if (fabsf(hf) >= 1.2e-38f && apq * apq > 1.0e-36 * fabs(app * aqq)) {
    const float th = df * __builtin_amdgcn_rcpf(hf);
    const float tf = copysignf(__builtin_amdgcn_rcpf(fabsf(th) + __builtin_amdgcn_sqrtf(fmaf(th, th, 1.0f))), th);
    t = (double)tf;
    const double f = fma(h, fma(t, t, -1.0), 2.0 * d * t);
    const float fp = 2.0f * fmaf(hf, tf, df);
    if (fabsf(fp) >= 1.2e-38f) t -= f * (double)__builtin_amdgcn_rcpf(fp);
    const double u = fma(t, t, 1.0);
    double y = (double)__builtin_amdgcn_rsqf((float)u);
    const double e = fma(-u, y * y, 1.0);
    c = fma(y * e, fma(e, 0.375, 0.5), y);
    sn = t * c;
  }
}

// The value of lane (lane ^ MASK) for the masks the cross rounds step by:
// data-parallel-primitive moves inside a row of 16 lanes, a lane exchange
// for 16.
template <int MASK>
__device__ __forceinline__ double lane_xor(double v) {
  if constexpr (MASK == 16) {
    return __shfl_xor(v, 16, 64);
  } else {
    constexpr int ctrl = MASK == 1 ? 0xB1 : MASK == 2 ? 0x4E : MASK == 7 ? 0x141 : 0x140;
    const int lo = __double2loint(v), hi = __double2hiint(v);
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, hi, ctrl, 0xF, 0xF, true),
                            __builtin_amdgcn_update_dpp(0, lo, ctrl, 0xF, 0xF, true));
  }
}

// Cross round R pairs local index k with 32 + (k ^ sigma(R)).  sigma walks
// all of 0..31 in Gray order over the basis 1, 2, 7, 15, 16, so that the
// partners of one round are those of the round before in the lane k ^ mask.
constexpr int cross_mask(int r) {  // sigma(r + 1) ^ sigma(r)
  return ((r + 1) & 1) ? 1 : ((r + 1) & 2) ? 2 : ((r + 1) & 4) ? 7 : ((r + 1) & 8) ? 15 : 16;
}
constexpr int cross_sigma(int r) {
  int s = 0;
  for (int i = 0; i < r; ++i) s ^= cross_mask(i);
  return s;
}

// A thread's share of the 64x64 problem through the cross rounds: the 2x2
// blocks (rows k, 32 + (k ^ sigma); columns k ^ d, 32 + (k ^ d ^ sigma)) for
// d = g and g + 16, and four rows of Q's columns k and 32 + (k ^ sigma).
struct CrossRegs {
  double ll[2], rr[2];   // S[k][k ^ d], S[32 + (k ^ sigma)][32 + (k ^ d ^ sigma)]
  double ql[4], qr[4];   // Q[4 g + j][k], Q[4 g + j][32 + (k ^ sigma)]
};

template <int R>
__device__ __forceinline__ void cross_round(double (*S)[SB], double2 (*rot)[32], double (*dgl)[SB], int k, int g,
                                            CrossRegs& v) {
  constexpr int SG = cross_sigma(R), b = R & 1;
  // keeps the compiler from computing all rounds' LDS addresses ahead of the
  // sweep loop, which spilled 35 registers
  asm volatile("" : "+v"(k));
  const double2 r1 = rot[b][k];
  const double c1 = r1.x, s1 = r1.y;
  double npq[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int k2 = k ^ (g + 16 * j);
    const double2 r2 = rot[b][k2];
    const double c2 = r2.x, s2 = r2.y;
    // S[q1][k2] is read from its mirror; the lane that owns the mirror is in
    // this wave and writes it after this read
    double* lr = &S[k][32 + (k2 ^ SG)];
    const double xpp = v.ll[j], xpq = *lr, xqp = S[k2][32 + (k ^ SG)], xqq = v.rr[j];
    const double rpp = c1 * xpp - s1 * xqp, rpq = c1 * xpq - s1 * xqq;
    const double rqp = s1 * xpp + c1 * xqp, rqq = s1 * xpq + c1 * xqq;
    v.ll[j] = c2 * rpp - s2 * rpq;
    npq[j] = s2 * rpp + c2 * rpq;
    v.rr[j] = s2 * rqp + c2 * rqq;
    *lr = npq[j];
  }
  if constexpr (R < 31) {
    // rotation k of the next round acts on S[k][32 + (k ^ SGN)], which is in
    // the block of d = SGN ^ SG
    constexpr int SGN = cross_sigma(R + 1), M = SG ^ SGN;
    if (g == (M & 15)) {
      const double apq = npq[M >> 4];
      const double dp = dgl[b][k], dq = dgl[b][32 + (k ^ SGN)];
      double c, sn, t;
      rotation_of(dp, dq, apq, c, sn, t);
      rot[b ^ 1][k] = make_double2(c, sn);
      dgl[b ^ 1][k] = dp - t * apq;
      dgl[b ^ 1][32 + (k ^ SGN)] = dq + t * apq;
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const double x = v.ql[j], y = v.qr[j];
    v.ql[j] = c1 * x - s1 * y;
    v.qr[j] = s1 * x + c1 * y;
  }
  if constexpr (R < 31) {
    constexpr int M = SG ^ cross_sigma(R + 1);
#pragma unroll
    for (int j = 0; j < 2; ++j) v.rr[j] = lane_xor<M>(v.rr[j]);
#pragma unroll
    for (int j = 0; j < 4; ++j) v.qr[j] = lane_xor<M>(v.qr[j]);
  }
  __syncthreads();
}

template <int... R>
__device__ __forceinline__ void cross_rounds(std::integer_sequence<int, R...>, double (*S)[SB], double2 (*rot)[32],
                                             double (*dgl)[SB], int k, int g, CrossRegs& v) {
  (cross_round<R>(S, rot, dgl, k, g, v), ...);
}

// The pair solve with cross rounds.  An inner sweep is, when intra[pair] is
// set, 31 rounds inside each 32-wide half (circle order on 32 indices, both
// halves at once), then 32 cross rounds, in which the 1024 index pairs
// across the two blocks are each rotated once.  The sweep schedule sets
// intra once per sweep of the block's group, so every index pair of the
// matrix is rotated once per sweep, in about half the sequential rounds of a
// full 64-index inner sweep.
//
// A cross round needs one barrier: the element that rotation k of the next
// round acts on is in a block of this round, whose thread computes the next
// angle right after its update, from the diagonals tracked in dgl
// (a - t apq, d + t apq per rotation), and publishes it in the other buffer.
// Of a block's four elements S[k][k2] stays in its thread's register and
// S[q1][q2] moves between lanes of the wave with the partners; S[k][q2] goes
// through LDS, and S[q1][k2] is read as its mirror.  Q's right columns move
// between lanes as well, so Q stays in registers.  A round then moves 36 KB
// through LDS; with all of S and Q's moving columns there it moved 112 KB,
// in 2-way bank conflicts.  S is stored with row stride 64: the rounds' XOR
// patterns put 16 consecutive lanes on 16 different bank pairs.
// Latency bound: 22 us a launch at 1020 orbitals (32 rounds, one workgroup per
// pair), 49 us before with two inner sweeps of 1.4 times longer rounds.
constexpr int CROSS_THREADS = 512;
__global__ __launch_bounds__(CROSS_THREADS) void k_jac_solve_x(
    const double* __restrict__ A, int lda, int nreal, const int* __restrict__ pairs,
    const int* __restrict__ intra, double* __restrict__ Qbuf, int* __restrict__ active, double tol,
    double skip_abs, int max_inner) {
  __shared__ double S[SB][SB];
  __shared__ double Q[SB][LDSW];
  __shared__ double2 rot[2][32];
  __shared__ double dgl[2][SB];
  __shared__ int rp[32], rq[32];
  __shared__ double red_off[CROSS_THREADS / 64], red_dg[CROSS_THREADS / 64];
  const int pidx = blockIdx.x;
  const int I = pairs[2 * pidx], J = pairs[2 * pidx + 1];
  const bool do_intra = intra[pidx] != 0;
  const int tid = threadIdx.x;
  const int k = tid & 31, g = tid >> 5;
  {
    // all loads of this thread in flight before the first LDS store; A is
    // symmetric, so column c of it is row c of S
    constexpr int PER = SB * SB / CROSS_THREADS;
    double v[PER];
#pragma unroll
    for (int it = 0; it < PER; ++it) {
      const int e = tid + CROSS_THREADS * it;
      v[it] = A[(size_t)gidx_dev(I, J, e % SB) + (size_t)gidx_dev(I, J, e / SB) * lda];
    }
#pragma unroll
    for (int it = 0; it < PER; ++it) {
      const int e = tid + CROSS_THREADS * it;
      S[e / SB][e % SB] = v[it];
    }
  }
  __syncthreads();
  CrossRegs v;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    v.ql[j] = (4 * g + j == k) ? 1.0 : 0.0;
    v.qr[j] = (4 * g + j == 32 + k) ? 1.0 : 0.0;
  }
  for (int sw = 0; sw < max_inner; ++sw) {
    double off = 0.0, dg = 0.0;
#pragma unroll
    for (int e = tid; e < SB * SB; e += CROSS_THREADS) {
      const int r = e / SB, c = e % SB;
      const double x = fabs(S[r][c]);
      if (r == c) {
        if (gidx_dev(I, J, r) < nreal) dg = fmax(dg, x);
      } else {
        off = fmax(off, x);
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
    for (int w = 0; w < CROSS_THREADS / 64; ++w) {
      off = fmax(off, red_off[w]);
      dg = fmax(dg, red_dg[w]);
    }
    __syncthreads();
    if (sw == 0 && off <= skip_abs) {
      if (tid == 0) active[pidx] = 0;
      return;
    }
    if (off <= tol * fmax(dg, 1.0)) break;
    if (do_intra) {
      // Q through LDS for these rounds
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        Q[4 * g + j][k] = v.ql[j];
        Q[4 * g + j][32 + k] = v.qr[j];
      }
      for (int round = 0; round < 31; ++round) {
        if (tid < 32) {
          // circle order on the 32 indices of half tid / 16
          const int h = tid >> 4, kk = tid & 15;
          auto pos = [&](int slot) { return slot == 0 ? 0 : 1 + ((slot - 1 + round) % 31); };
          int p = 32 * h + pos(kk), q = 32 * h + pos(31 - kk);
          if (p > q) { const int x = p; p = q; q = x; }
          double c, sn, t;
          rotation_of(S[p][p], S[q][q], S[p][q], c, sn, t);
          rot[0][tid] = make_double2(c, sn);
          rp[tid] = p;
          rq[tid] = q;
        }
        __syncthreads();
        const double2 r2 = rot[0][k];
        const int p2 = rp[k], q2 = rq[k];
        const double c2 = r2.x, s2 = r2.y;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int k1 = g + 16 * j;
          const double2 r1 = rot[0][k1];
          const int p1 = rp[k1], q1 = rq[k1];
          const double c1 = r1.x, s1 = r1.y;
          const double xpp = S[p1][p2], xpq = S[p1][q2], xqp = S[q1][p2], xqq = S[q1][q2];
          const double rpp = c1 * xpp - s1 * xqp, rpq = c1 * xpq - s1 * xqq;
          const double rqp = s1 * xpp + c1 * xqp, rqq = s1 * xpq + c1 * xqq;
          S[p1][p2] = c2 * rpp - s2 * rpq;
          S[p1][q2] = s2 * rpp + c2 * rpq;
          S[q1][p2] = c2 * rqp - s2 * rqq;
          S[q1][q2] = s2 * rqp + c2 * rqq;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int row = 4 * g + j;
          const double x = Q[row][p2], y = Q[row][q2];
          Q[row][p2] = c2 * x - s2 * y;
          Q[row][q2] = s2 * x + c2 * y;
        }
        __syncthreads();
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v.ql[j] = Q[4 * g + j][k];
        v.qr[j] = Q[4 * g + j][32 + k];
      }
    }
    // cross rounds: angles of round 0 and the diagonals after it
    if (tid < 32) {
      const int p = tid, q = 32 + tid;
      const double app = S[p][p], aqq = S[q][q], apq = S[p][q];
      double c, sn, t;
      rotation_of(app, aqq, apq, c, sn, t);
      rot[0][tid] = make_double2(c, sn);
      dgl[0][p] = app - t * apq;
      dgl[0][q] = aqq + t * apq;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      v.ll[j] = S[k][k ^ (g + 16 * j)];
      v.rr[j] = S[32 + k][32 + (k ^ (g + 16 * j))];
    }
    __syncthreads();
    cross_rounds(std::make_integer_sequence<int, 32>{}, S, rot, dgl, k, g, v);
    // Q's right columns back in order, and S whole again for another sweep
    constexpr int SL = cross_sigma(31);
#pragma unroll
    for (int j = 0; j < 4; ++j) v.qr[j] = __shfl(v.qr[j], (tid & 32) | (k ^ SL), 64);
    if (sw + 1 < max_inner) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int d = g + 16 * j;
        S[k][k ^ d] = v.ll[j];
        S[32 + (k ^ SL)][32 + (k ^ d ^ SL)] = v.rr[j];
        S[32 + k][k ^ d] = S[k ^ d][32 + k];
      }
      __syncthreads();
    }
  }
  // to LDS, then out with consecutive lanes on consecutive rows
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    Q[4 * g + j][k] = v.ql[j];
    Q[4 * g + j][32 + k] = v.qr[j];
  }
  __syncthreads();
  double* Qo = Qbuf + (size_t)pidx * SB * SB;
#pragma unroll
  for (int e = tid; e < SB * SB; e += CROSS_THREADS) Qo[e] = Q[e % SB][e / SB];
  if (tid == 0) active[pidx] = 1;
}

__device__ __forceinline__ int gidx(int pairI, int pairJ, int local) {
  return (local < BS) ? pairI * BS + local : pairJ * BS + (local - BS);
}

// Tile t -> pair indices P1 <= P2.  The pairs [0, npo) and [npo, npairs) form
// two groups (npo == npairs: one group); tiles across the groups are not
// enumerated, since the grouped schedule never couples them.
__device__ __forceinline__ void tri_of(int t, int& P1, int& P2) {
  P2 = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
  while ((P2 + 1) * (P2 + 2) / 2 <= t) ++P2;
  while (P2 * (P2 + 1) / 2 > t) --P2;
  P1 = t - P2 * (P2 + 1) / 2;
}
__device__ __forceinline__ void tile_of(int t, int npairs, int npo, int& P1, int& P2) {
  (void)npairs;
  const int t0 = npo * (npo + 1) / 2;
  if (t < t0) {
    tri_of(t, P1, P2);
  } else {
    tri_of(t - t0, P1, P2);
    P1 += npo;
    P2 += npo;
  }
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


// This thread's 8 elements (e = tid + 512 it) of a 64x64 rotation, all
// loads issued together; Q = I for a pair marked inactive.
constexpr int UPD_NT = 512;  // eight waves per update workgroup
__device__ __forceinline__ void stage_q(double (&v)[SB * SB / UPD_NT], const double* __restrict__ q, bool active,
                                        int tid) {
  if (active) {
#pragma unroll
    for (int it = 0; it < SB * SB / UPD_NT; ++it) v[it] = q[tid + UPD_NT * it];
  } else {
#pragma unroll
    for (int it = 0; it < SB * SB / UPD_NT; ++it) {
      const int e = tid + UPD_NT * it;
      v[it] = (e % SB == e / SB) ? 1.0 : 0.0;
    }
  }
}

// MFMA versions of the two update kernels (same data flow as above).
__global__ __launch_bounds__(UPD_NT) void k_jac_apply_a_mfma(double* __restrict__ A, int lda,
                                                          int npairs, int npo,
                                                          const int* __restrict__ pairs,
                                                          const double* __restrict__ Qbuf,
                                                          const int* __restrict__ active) {
  int P1, P2;
  tile_of(blockIdx.x, npairs, npo, P1, P2);
  const bool a1 = active[P1] != 0, a2 = active[P2] != 0;
  if (!a1 && !a2) return;
  // two 64 x 65 LDS tiles (66.5 KB) so two workgroups fit on a CU: the tile of
  // A, then Q1^T A, then the result; Q1, then Q2
  __shared__ double At[SB][LDSW];
  __shared__ double Qs[SB][LDSW];
  const int I1 = pairs[2 * P1], J1 = pairs[2 * P1 + 1];
  const int I2 = pairs[2 * P2], J2 = pairs[2 * P2 + 1];
  const int tid = threadIdx.x;
  const double* q1 = Qbuf + (size_t)P1 * SB * SB;
  const double* q2 = Qbuf + (size_t)P2 * SB * SB;
  // every global load of a stage is issued before the first LDS store, so a
  // thread waits for memory once per stage, not once per element; Q2 is
  // fetched into registers now and lands in LDS after the first product
  constexpr int PER = SB * SB / UPD_NT;  // element e = tid + 512 it: row tid % 64, column tid / 64 + 8 it
  double va[PER], vq[PER], vq2[PER];
#pragma unroll
  for (int it = 0; it < PER; ++it) {
    const int e = tid + UPD_NT * it;
    va[it] = A[(size_t)gidx(I1, J1, e % SB) + (size_t)gidx(I2, J2, e / SB) * lda];
  }
  stage_q(vq, q1, a1, tid);
  if (P1 != P2) stage_q(vq2, q2, a2, tid);
#pragma unroll
  for (int it = 0; it < PER; ++it) {
    const int e = tid + UPD_NT * it;
    At[e % SB][e / SB] = va[it];
    Qs[e % SB][e / SB] = vq[it];
  }
  __syncthreads();
  d4_t acc[2];
  for (int i = 0; i < 2; ++i) acc[i] = d4_t{0.0, 0.0, 0.0, 0.0};
  mfma_tile64_w8([&](int r, int k) { return Qs[k][r]; }, [&](int k, int c) { return At[k][c]; }, SB, acc);
  __syncthreads();
  mfma_tile64_w8_store(acc, [&](int r, int c, double v) { At[r][c] = v; });
  if (P1 != P2) {
#pragma unroll
    for (int it = 0; it < PER; ++it) {
      const int e = tid + UPD_NT * it;
      Qs[e % SB][e / SB] = vq2[it];
    }
  }
  __syncthreads();
  for (int i = 0; i < 2; ++i) acc[i] = d4_t{0.0, 0.0, 0.0, 0.0};
  mfma_tile64_w8([&](int r, int k) { return At[r][k]; }, [&](int k, int c) { return Qs[k][c]; }, SB, acc);
  // stage the result in LDS and write both the tile and its mirror with
  // consecutive lanes on consecutive rows of A
  __syncthreads();
  mfma_tile64_w8_store(acc, [&](int r, int c, double v) { At[r][c] = v; });
  __syncthreads();
  if (P1 == P2) {
    for (int e = tid; e < SB * SB; e += UPD_NT) {
      const int r = e % SB, c = e / SB;
      const double v = (r == c) ? At[r][c] : 0.5 * (At[r][c] + At[c][r]);
      A[(size_t)gidx(I1, J1, r) + (size_t)gidx(I2, J2, c) * lda] = v;
    }
    return;
  }
  for (int e = tid; e < SB * SB; e += UPD_NT) {
    const int r = e % SB, c = e / SB;
    A[(size_t)gidx(I1, J1, r) + (size_t)gidx(I2, J2, c) * lda] = At[r][c];
  }
  for (int e = tid; e < SB * SB; e += UPD_NT) {
    const int c = e % SB, r = e / SB;
    A[(size_t)gidx(I2, J2, c) + (size_t)gidx(I1, J1, r) * lda] = At[r][c];
  }
}

__global__ __launch_bounds__(UPD_NT) void k_jac_apply_c_mfma(double* __restrict__ C, int ldc, int nrows,
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
  constexpr int PER = SB * SB / UPD_NT;
  double vc[PER], vq[PER];
  {
    const int gr = row0 + tid % SB;  // the same row for all of this thread's elements
#pragma unroll
    for (int it = 0; it < PER; ++it) {
      const int e = tid + UPD_NT * it;
      vc[it] = (gr < nrows) ? C[(size_t)gr + (size_t)gidx(I, J, e / SB) * ldc] : 0.0;
    }
  }
  stage_q(vq, q, true, tid);
#pragma unroll
  for (int it = 0; it < PER; ++it) {
    const int e = tid + UPD_NT * it;
    Ct[e % SB][e / SB] = vc[it];
    Qs[e % SB][e / SB] = vq[it];
  }
  __syncthreads();
  d4_t acc[2];
  for (int i = 0; i < 2; ++i) acc[i] = d4_t{0.0, 0.0, 0.0, 0.0};
  mfma_tile64_w8([&](int r, int k) { return Ct[r][k]; }, [&](int k, int c) { return Qs[k][c]; }, SB, acc);
  // stage in LDS, then store with consecutive lanes on consecutive rows of C
  __syncthreads();
  mfma_tile64_w8_store(acc, [&](int r, int c, double v) { Ct[r][c] = v; });
  __syncthreads();
  for (int e = tid; e < SB * SB; e += UPD_NT) {
    const int r = e % SB, c = e / SB;
    const int gr = row0 + r;
    if (gr < nrows) C[(size_t)gr + (size_t)gidx(I, J, c) * ldc] = Ct[r][c];
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
                                                       double* __restrict__ out) {
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
    out[0] = r1[0];
    out[1] = r2[0];
  }
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

// Stable ascending rank sort of the diagonal; perm[rank] = index.  One
// thread per entry across the grid; the diagonal goes through LDS in chunks.
constexpr int SORT_CHUNK = 2048;
__global__ __launch_bounds__(256) void k_sort_diag(int npad, const double* __restrict__ A, int lda,
                                                   int* __restrict__ perm, double* __restrict__ eig) {
  __shared__ double d[SORT_CHUNK];
  const int i = blockIdx.x * 256 + threadIdx.x;
  const double di = (i < npad) ? A[(size_t)i + (size_t)i * lda] : 0.0;
  int rank = 0;
  for (int j0 = 0; j0 < npad; j0 += SORT_CHUNK) {
    const int nj = min(SORT_CHUNK, npad - j0);
    for (int j = threadIdx.x; j < nj; j += 256) d[j] = A[(size_t)(j0 + j) + (size_t)(j0 + j) * lda];
    __syncthreads();
    for (int j = 0; j < nj; ++j) {
      const double dj = d[j];
      rank += (dj < di) || (dj == di && j0 + j < i);
    }
    __syncthreads();
  }
  if (i < npad) {
    perm[rank] = i;
    eig[rank] = di;
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
  // buffers below may be re-allocated: no C update of an earlier solve may
  // still be reading them
  if (cstream) MHIP_CHECK(hipStreamSynchronize(cstream));
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
  qbuf.ensure((size_t)nsteps * npairs * SB * SB * sizeof(double));
  part.ensure((size_t)2 * npad * sizeof(double) + 64);
  perm.ensure((size_t)npad * sizeof(int));
  active.ensure((size_t)nsteps * npairs * sizeof(int));
  if (!cstream) MHIP_CHECK(hipStreamCreateWithFlags(&cstream, hipStreamNonBlocking));
  if (!ev_join) MHIP_CHECK(hipEventCreateWithFlags(&ev_join, hipEventDisableTiming));
  while ((int)ev_solved.size() < nsteps) {
    hipEvent_t a, b;
    MHIP_CHECK(hipEventCreateWithFlags(&a, hipEventDisableTiming));
    MHIP_CHECK(hipEventCreateWithFlags(&b, hipEventDisableTiming));
    ev_solved.push_back(a);
    ev_cdone.push_back(b);
  }
  cdone_pending.assign(ev_cdone.size(), 0);
  counts.ensure((size_t)2 * nb * sizeof(int));
}

void jacobi_set_identity(hipStream_t s, int npad, double* C, int ldc) {
  hipLaunchKernelGGL(k_set_identity, dim3((npad + 255) / 256, npad), dim3(256), 0, s, npad, C, ldc);
  MHIP_LAUNCH_CHECK();
}

int jacobi_sweeps(hipStream_t s, JacobiPlan& plan, double* A, double* C, double tol, int max_sweeps,
                  double* host_scal, double* dev_scal, int* sweeps_done) {
  const int lda = plan.npad;
  int done = 0;
  hipStream_t cs = plan.cstream;
  // Inner sweeps per step.  Cross schedule: one; a second saves up to a fifth
  // of the sweeps (54 instead of 66 in the plain SCF of 1020 orbitals) for
  // twice the rounds (109 ms instead of 102; 16.6 instead of 15.2 ms at 174
  // orbitals).  A matrix that is one pair problem is solved in one launch.
  const bool cross = g_jacobi_schedule == 1;
  const int inner = plan.max_inner > 0 ? plan.max_inner : !cross ? 2 : plan.npairs == 1 ? 16 : 1;
  const double inner_tol = plan.npairs == 1 ? 0.5 * tol : 1.0e-14;
  // the C updates start after whatever the caller queued on C
  MHIP_CHECK(hipEventRecord(plan.ev_join, s));
  MHIP_CHECK(hipStreamWaitEvent(cs, plan.ev_join, 0));
  // and the caller's later work on C waits for the last of them
  auto join = [&] {
    MHIP_CHECK(hipEventRecord(plan.ev_join, cs));
    MHIP_CHECK(hipStreamWaitEvent(s, plan.ev_join, 0));
  };
  for (int sw = 0; sw <= max_sweeps; ++sw) {
    hipLaunchKernelGGL(k_offmax_partial, dim3(plan.n), dim3(256), 0, s, plan.n, A, lda,
                       plan.grouped ? plan.split : 0, plan.part.as<double>());
    MHIP_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_offmax_final, dim3(1), dim3(1024), 0, s, plan.n, plan.part.as<double>(),
                       dev_scal);
    MHIP_LAUNCH_CHECK();
    MHIP_CHECK(hipMemcpyAsync(host_scal, dev_scal, 2 * sizeof(double), hipMemcpyDeviceToHost, s));
    MHIP_CHECK(hipStreamSynchronize(s));
    const double thr = tol * std::max(1.0, host_scal[1]);
    if (host_scal[0] <= thr) break;
    // pairs whose whole 64x64 block is already this diagonal are left alone
    const double skip_abs = 0.1 * thr;
    if (sw == max_sweeps) {
      join();
      if (sweeps_done) *sweeps_done = done;
      return 1;
    }
    const int nsteps = plan.nsteps;
    if (plan.timing && plan.ev.size() < (size_t)(6 * nsteps)) {
      for (auto e : plan.ev) (void)hipEventDestroy(e);
      plan.ev.assign(6 * nsteps, nullptr);
      for (auto& e : plan.ev) MHIP_CHECK(hipEventCreate(&e));
    }
    const int npv = plan.npairs - plan.npo;
    const int ntiles = plan.npo * (plan.npo + 1) / 2 + npv * (npv + 1) / 2;
    for (int step = 0; step < nsteps; ++step) {
      const int* pr = plan.pairs.as<int>() + (size_t)step * plan.npairs * 2;
      double* q = plan.qbuf.as<double>() + (size_t)step * plan.npairs * SB * SB;
      int* act = plan.active.as<int>() + (size_t)step * plan.npairs;
      // the slot's previous C update (one sweep earlier) must have read it
      if (plan.cdone_pending[step]) MHIP_CHECK(hipStreamWaitEvent(s, plan.ev_cdone[step], 0));
      if (plan.timing) MHIP_CHECK(hipEventRecord(plan.ev[6 * step + 0], s));
      if (g_jacobi_schedule == 1) {
        const int* fl = plan.intra.as<int>() + (size_t)step * plan.npairs;
        hipLaunchKernelGGL(k_jac_solve_x, dim3(plan.npairs), dim3(CROSS_THREADS), 0, s, A, lda, plan.n, pr, fl,
                           q, act, inner_tol, skip_abs, inner);
      } else {
        hipLaunchKernelGGL(k_jac_solve, dim3(plan.npairs), dim3(SOLVE_THREADS), 0, s, A, lda, plan.n, pr, q,
                           act, 1.0e-14, skip_abs, inner);
      }
      MHIP_LAUNCH_CHECK();
      if (plan.timing) {
        MHIP_CHECK(hipEventRecord(plan.ev[6 * step + 1], s));
        hipLaunchKernelGGL(k_count_active, dim3(1), dim3(64), 0, s, plan.npairs, plan.npo, act,
                           plan.counts.as<int>() + 2 * step);
      }
      if (g_kernel_variant == 1) {
        if (plan.timing) MHIP_CHECK(hipEventRecord(plan.ev[6 * step + 2], s));
        hipLaunchKernelGGL(k_jac_apply_a_mfma, dim3(ntiles), dim3(UPD_NT), 0, s, A, lda, plan.npairs, plan.npo, pr, q,
                           act);
        MHIP_LAUNCH_CHECK();
        if (plan.timing) MHIP_CHECK(hipEventRecord(plan.ev[6 * step + 3], s));
        // C <- C Q on the side stream once this step's A update is done, so
        // it overlaps the next step's pair solves, which leave most CUs idle
        MHIP_CHECK(hipEventRecord(plan.ev_solved[step], s));
        MHIP_CHECK(hipStreamWaitEvent(cs, plan.ev_solved[step], 0));
        if (plan.timing) MHIP_CHECK(hipEventRecord(plan.ev[6 * step + 4], cs));
        hipLaunchKernelGGL(k_jac_apply_c_mfma, dim3(plan.npad / SB, plan.npairs), dim3(UPD_NT), 0, cs, C, lda,
                           plan.npad, pr, q, act);
        MHIP_LAUNCH_CHECK();
        if (plan.timing) MHIP_CHECK(hipEventRecord(plan.ev[6 * step + 5], cs));
      } else {
        hipLaunchKernelGGL(k_jac_apply_a, dim3(ntiles), dim3(256), 0, s, A, lda, plan.npairs, plan.npo, pr, q,
                           act);
        MHIP_LAUNCH_CHECK();
        MHIP_CHECK(hipEventRecord(plan.ev_solved[step], s));
        MHIP_CHECK(hipStreamWaitEvent(cs, plan.ev_solved[step], 0));
        hipLaunchKernelGGL(k_jac_apply_c, dim3(plan.npad / SB, plan.npairs), dim3(256), 0, cs, C, lda,
                           plan.npad, pr, q, act);
        MHIP_LAUNCH_CHECK();
      }
      MHIP_CHECK(hipEventRecord(plan.ev_cdone[step], cs));
      plan.cdone_pending[step] = 1;
    }
    if (plan.timing && g_kernel_variant == 1) {
      MHIP_CHECK(hipStreamSynchronize(cs));
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
          if (first >= plan.npairs) continue;
          const long long per =
              g_jacobi_schedule == 1
                  ? 1024 + (plan.intra_host[(size_t)step * plan.npairs + first] ? 992 : 0)
                  : 2016LL * inner;
          plan.active_rotations += per * act[2 * step + g];
        }
        plan.active_tiles += (long long)ntiles - u0 * (u0 + 1) / 2 - u1 * (u1 + 1) / 2;
        float a = 0.f, b = 0.f, c2 = 0.f;
        MHIP_CHECK(hipEventElapsedTime(&a, plan.ev[6 * step + 0], plan.ev[6 * step + 1]));
        MHIP_CHECK(hipEventElapsedTime(&b, plan.ev[6 * step + 2], plan.ev[6 * step + 3]));
        MHIP_CHECK(hipEventElapsedTime(&c2, plan.ev[6 * step + 4], plan.ev[6 * step + 5]));
        plan.t_solve_ms += a;
        plan.t_apply_ms += b;
        plan.t_applyc_ms += c2;
        plan.n_solve++;
        plan.n_apply++;
        plan.n_applyc++;
      }
    }
    ++done;
  }
  join();
  if (sweeps_done) *sweeps_done = done;
  return 0;
}

void jacobi_sort(hipStream_t s, JacobiPlan& plan, const double* A, const double* C, double* Cout,
                 double* eig_dev) {
  const int npad = plan.npad;
  hipLaunchKernelGGL(k_sort_diag, dim3((npad + 255) / 256), dim3(256), 0, s, npad, A, npad, plan.perm.as<int>(),
                     eig_dev);
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
