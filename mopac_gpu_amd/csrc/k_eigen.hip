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

// Rotation by the smaller of the angles that zero apq in [[app, apq], [apq,
// aqq]]: with d = aqq - app, h = 2 apq and r = sqrt(d^2 + h^2), c^2 = (1 +
// |d| / r) / 2 and s = sign(d) h / (2 r c); t = s / c, and the diagonal after
// it is app - t apq, aqq + t apq.  c and s start in FP32 (a reciprocal square
// root is one instruction there), an FP64 step turns them by what they leave
// of apq (angle good to about 1e-14), and they are scaled to c^2 + s^2 = 1 in
// FP64 to the last bit.  Every round of a pair solve waits for this chain of
// 17 dependent operations; FP64 division and square roots take 100.  With
// apq and d both below 1e-15, far under any stopping threshold (they are
// absolute), nothing is turned.
__device__ __forceinline__ void rotation_of(double app, double aqq, double apq, double& c, double& sn,
                                            double& t) {
  const double d = aqq - app;
  const float df = (float)d, ad = fabsf(df), hh = (float)apq;
  const float r2 = fmaf(4.0f * hh, hh, ad * ad);
  const float rinv = __builtin_amdgcn_rsqf(r2);
  const float c2 = fmaf(0.5f * ad, rinv, 0.5f);
  const float cinv = __builtin_amdgcn_rsqf(c2);
  const bool none = r2 < 1.0e-30f;
  const float cf = none ? 1.0f : c2 * cinv, sf = none ? 0.0f : copysignf(1.0f, df) * hh * rinv * cinv;
  double c0 = (double)cf, s0 = (double)sf;
  // the off-diagonal element after the rotation, over sign(d) r
  const double left = fma(fma(c0, c0, -s0 * s0), apq, -(c0 * s0) * d);
  const double turn = left * (double)(none ? 0.0f : copysignf(rinv, df));
  const double c1 = fma(-turn, s0, c0), s1 = fma(turn, c0, s0);
  const double e = fma(-c1, c1, fma(-s1, s1, 1.0));
  const double corr = fma(e, fma(e, 0.375, 0.5), 1.0);
  c = c1 * corr;
  sn = s1 * corr;
  const double ci = none ? 1.0 : (double)cinv;
  t = sn * (ci * fma(-c, ci, 2.0));  // s / c, 1 / c by a Newton step from FP32's
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

// A thread's share of the 64x64 problem through the cross rounds: one 2x2
// block (rows k, q = 32 + (k ^ sigma); columns k ^ d, 32 + (k ^ d ^ sigma)),
// and four rows of Q's columns k and q.  k is the lane in its half-wave g.
// S is symmetric, so of the blocks (k, k ^ d) and (k ^ d, k) only one is
// kept: the one whose k has the highest bit of d equal to d's lowest bit
// (d > 1), which lets d and d + 1 share a half-wave.  d = 1 has a half-wave
// to itself with both kept; the diagonal blocks (d = 0) are the rotated pairs
// themselves, whose diagonals dgl tracks and whose off-diagonal becomes 0.
struct CrossRegs {
  double ll, rr;         // S[k][k ^ d], S[32 + (k ^ sigma)][32 + (k ^ d ^ sigma)]
  double ql[4], qr[4];   // Q[4 g + j][k], Q[4 g + j][32 + (k ^ sigma)], a round behind
  double c, s;           // the rotation Q has still to take
  int d, top;            // top: the highest bit of d; 0 where both blocks are kept
  int own_rot, mate_rot; // LDS byte offsets of rot[0][k], rot[0][k ^ d]
  int lr, rl;            // and of S[k][32 + (k ^ d)], S[k ^ d][32 + k]
  int own_q;             // and of dgl[0][32 + k]
};

__device__ __forceinline__ void cross_setup(CrossRegs& v, int k, int g) {
  if (g < 8) { v.top = 16; v.d = 16 + 2 * g + ((k >> 4) & 1); }
  else if (g < 12) { v.top = 8; v.d = 8 + 2 * (g - 8) + ((k >> 3) & 1); }
  else if (g < 14) { v.top = 4; v.d = 4 + 2 * (g - 12) + ((k >> 2) & 1); }
  else if (g < 15) { v.top = 2; v.d = 2 + ((k >> 1) & 1); }
  else { v.top = 0; v.d = 1; }
  const int k2 = k ^ v.d;
  v.own_rot = k * 16;
  v.mate_rot = k2 * 16;
  v.lr = (k * SB + 32 + k2) * 8;
  v.rl = (k2 * SB + 32 + k) * 8;
  v.own_q = (32 + k) * 8;
}

__device__ __forceinline__ void cross_turn_q(CrossRegs& v) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const double x = v.ql[j], y = v.qr[j];
    v.ql[j] = v.c * x - v.s * y;
    v.qr[j] = v.s * x + v.c * y;
  }
}

template <class T>
__device__ __forceinline__ T& lds_at(void* base, int off) {
  return *reinterpret_cast<T*>(static_cast<char*>(base) + off);
}

// the half-wave that holds d = mask
constexpr int mask_group(int m) { return m == 1 ? 15 : m == 2 ? 14 : m == 7 ? 13 : m == 15 ? 11 : 0; }

template <int R>
__device__ __forceinline__ void cross_round(double (*S)[SB], double2 (*rot)[32], double (*dgl)[SB], int k, int g,
                                            CrossRegs& v) {
  constexpr int SG = cross_sigma(R), b = R & 1;
  // rotation k of the next round acts on S[k][32 + (k ^ SGN)], which is in
  // this round's block of d = M
  constexpr int SGN = R < 31 ? cross_sigma(R + 1) : 0, M = R < 31 ? SG ^ SGN : 0;
  // keeps the compiler from computing all rounds' LDS addresses ahead of the
  // sweep loop, which spilled registers
  asm volatile("" : "+v"(v.lr), "+v"(v.rl), "+v"(v.own_q));
  const int lr = v.lr ^ (SG * 8), rl = v.rl ^ (SG * 8), nq = v.own_q ^ (SGN * 8);
  const double2 r1 = lds_at<double2>(rot[b], v.own_rot), r2 = lds_at<double2>(rot[b], v.mate_rot);
  const double xpq = lds_at<double>(S, lr), xqp = lds_at<double>(S, rl);
  const double dp = dgl[b][k], dq = lds_at<double>(dgl[b], nq);
  // while those arrive: Q's turn of the round before, and its partners
  if constexpr (R > 0) {
    constexpr int MP = cross_sigma(R - 1) ^ SG;
    cross_turn_q(v);
#pragma unroll
    for (int j = 0; j < 4; ++j) v.qr[j] = lane_xor<MP>(v.qr[j]);
  }
  const double c1 = r1.x, s1 = r1.y, c2 = r2.x, s2 = r2.y;
  v.c = c1;
  v.s = s1;
  const double xpp = v.ll, xqq = v.rr;
  const double rpp = c1 * xpp - s1 * xqp, rpq = c1 * xpq - s1 * xqq;
  const double rqp = s1 * xpp + c1 * xqp, rqq = s1 * xpq + c1 * xqq;
  const double npq = s2 * rpp + c2 * rpq, nqp = c2 * rqp - s2 * rqq;
  v.ll = c2 * rpp - s2 * rpq;
  v.rr = s2 * rqp + c2 * rqq;
  // the next round's pairs are zero after it, and not read in it
  const bool next_pair = R < 31 && v.d == M;
  lds_at<double>(S, lr) = next_pair ? 0.0 : npq;
  lds_at<double>(S, rl) = next_pair ? 0.0 : nqp;
  if constexpr (R < 31) {
    if (g == mask_group(M)) {
      // lane k of the half-wave takes rotation k: where the block kept is
      // that of k ^ M, its S[q1][k2]
      const double other = lane_xor<M>(nqp);
      const double apq = v.d == M ? npq : other;
      double c, sn, t;
      rotation_of(dp, dq, apq, c, sn, t);
      lds_at<double2>(rot[b ^ 1], v.own_rot) = make_double2(c, sn);
      dgl[b ^ 1][k] = dp - t * apq;
      lds_at<double>(dgl[b ^ 1], nq) = dq + t * apq;
    }
    // S[q1][q2] of the partners to come, from lane k ^ M, or from its mirror
    // where that lane keeps the other block
    if constexpr (M == 16) {
      v.rr = __shfl(v.rr, (threadIdx.x & 32) | (k ^ 16 ^ (v.top == 16 ? v.d : 0)), 64);
    } else if constexpr (M == 1) {
      v.rr = lane_xor<1>(v.rr);
    } else {
      constexpr int first = M == 2 ? 14 : M == 7 ? 12 : 8;  // half-waves from here on may turn
      if (g >= first)
        v.rr = __shfl(v.rr, (threadIdx.x & 32) | (k ^ M ^ ((v.top & M) ? v.d : 0)), 64);
      else
        v.rr = lane_xor<M>(v.rr);
    }
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
// S[q1][q2] moves between lanes of the wave with the partners; S[k][q2] and
// S[q1][k2] = S[k2][q1] go through LDS.  Q's right columns move between lanes
// as well, so Q stays in registers, and its turn waits for the next round's
// loads.  With all of S and Q's moving columns in LDS a round moved 112 KB
// through it, in 2-way bank conflicts; now 38 KB.  S is stored with row
// stride 64: the rounds' XOR patterns put 16 consecutive lanes on 16
// different bank pairs.
constexpr int CROSS_THREADS = 512;

// LDS of one workgroup of the cross schedule: two 64 x 65 tiles, shared by
// the pair solve (S with stride 64, then Q or its two operand halves) and
// the update tiles.
struct JacLds {
  double m[2 * SB * LDSW];
  double2 rot[2][32];
  double dgl[2][SB];
  int rp[32], rq[32];
  double red_off[CROSS_THREADS / 64], red_dg[CROSS_THREADS / 64];
  __device__ double (*s())[SB] { return reinterpret_cast<double (*)[SB]>(m); }
  __device__ double (*q())[LDSW] { return reinterpret_cast<double (*)[LDSW]>(m + SB * SB); }
};

// What a pair solve reads besides its 64x64 problem and what it writes.
struct JacSolve {
  int nreal;
  double* q;      // 64 x 64 rotation, column-major
  int* active;
  double* di;     // the two 32 x 32 diagonal blocks after the solve (may be null)
  double* dj;
  double tol, skip_abs;
  int max_inner;
};

// Diagonalizes the problem in lds.s(): the upper right quadrant and the two
// diagonal ones, and the lower left one where do_intra asks for it.
__device__ __forceinline__ void pair_solve(JacLds& lds, int I, int J, bool do_intra, const JacSolve& p) {
  double(*S)[SB] = lds.s();
  double(*Q)[LDSW] = lds.q();
  const int tid = threadIdx.x;
  const int k = tid & 31, g = tid >> 5;
  CrossRegs v;
  cross_setup(v, k, g);
  const int k2 = k ^ v.d;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    v.ql[j] = (4 * g + j == k) ? 1.0 : 0.0;
    v.qr[j] = (4 * g + j == 32 + k) ? 1.0 : 0.0;
  }
  bool rotated = false;
  for (int sw = 0; sw < p.max_inner; ++sw) {
    v.ll = S[k][k2];
    v.rr = S[32 + k][32 + k2];
    double off = fmax(fabs(v.ll), fabs(v.rr)), dg = 0.0;
    off = fmax(off, fmax(fabs(S[g][32 + k]), fabs(S[16 + g][32 + k])));
    if (tid < SB && gidx_dev(I, J, tid) < p.nreal) dg = fabs(S[tid][tid]);
    off = wave_max(off);
    dg = wave_max(dg);
    if ((tid & 63) == 0) {
      lds.red_off[tid >> 6] = off;
      lds.red_dg[tid >> 6] = dg;
    }
    __syncthreads();
    off = 0.0;
    dg = 0.0;
#pragma unroll
    for (int w = 0; w < CROSS_THREADS / 64; ++w) {
      off = fmax(off, lds.red_off[w]);
      dg = fmax(dg, lds.red_dg[w]);
    }
    __syncthreads();
    if ((sw == 0 && off <= p.skip_abs) || off <= p.tol * fmax(dg, 1.0)) break;
    rotated = true;
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
          int a = 32 * h + pos(kk), b = 32 * h + pos(31 - kk);
          if (a > b) { const int x = a; a = b; b = x; }
          double c, sn, t;
          rotation_of(S[a][a], S[b][b], S[a][b], c, sn, t);
          lds.rot[0][tid] = make_double2(c, sn);
          lds.rp[tid] = a;
          lds.rq[tid] = b;
        }
        __syncthreads();
        const double2 r2 = lds.rot[0][k];
        const int p2 = lds.rp[k], q2 = lds.rq[k];
        const double c2 = r2.x, s2 = r2.y;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int k1 = g + 16 * j;
          const double2 r1 = lds.rot[0][k1];
          const int p1 = lds.rp[k1], q1 = lds.rq[k1];
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
      v.ll = S[k][k2];
      v.rr = S[32 + k][32 + k2];
    }
    // cross rounds: angles of round 0 and the diagonals after it
    if (tid < 32) {
      const double app = S[tid][tid], aqq = S[32 + tid][32 + tid], apq = S[tid][32 + tid];
      double c, sn, t;
      rotation_of(app, aqq, apq, c, sn, t);
      S[tid][32 + tid] = 0.0;
      lds.rot[0][tid] = make_double2(c, sn);
      lds.dgl[0][tid] = app - t * apq;
      lds.dgl[0][32 + tid] = aqq + t * apq;
    }
    __syncthreads();
    cross_rounds(std::make_integer_sequence<int, 32>{}, S, lds.rot, lds.dgl, k, g, v);
    cross_turn_q(v);
    // the moving columns back in order, and S whole again for another sweep
    constexpr int SL = cross_sigma(31);
#pragma unroll
    for (int j = 0; j < 4; ++j) v.qr[j] = __shfl(v.qr[j], (tid & 32) | (k ^ SL), 64);
    // S whole again: the diagonal blocks here, the upper right one is there
    const int last = 32 + (k ^ SL), last2 = 32 + (k2 ^ SL);
    S[k][k2] = S[k2][k] = v.ll;
    S[last][last2] = S[last2][last] = v.rr;
    if (tid < SB) S[tid][tid] = lds.dgl[1][tid];
    __syncthreads();
    if (do_intra && sw + 1 < p.max_inner) {
      S[32 + k][g] = S[g][32 + k];
      S[32 + k][16 + g] = S[16 + g][32 + k];
      __syncthreads();
    }
  }
  if (p.di) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int e = (g + 16 * j) * BS + k;
      p.di[e] = S[g + 16 * j][k];
      p.dj[e] = S[32 + g + 16 * j][32 + k];
    }
  }
  if (tid == 0) *p.active = rotated ? 1 : 0;
  if (!rotated) return;
  // Q to LDS, then out with consecutive lanes on consecutive rows
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    Q[4 * g + j][k] = v.ql[j];
    Q[4 * g + j][32 + k] = v.qr[j];
  }
  __syncthreads();
#pragma unroll
  for (int e = tid; e < SB * SB; e += CROSS_THREADS) p.q[e] = Q[e % SB][e / SB];
}

// The pair solve on a matrix in memory.
__global__ __launch_bounds__(CROSS_THREADS, 4) void k_jac_solve_x(
    const double* __restrict__ A, int lda, int nreal, const int* __restrict__ pairs,
    const int* __restrict__ intra, double* __restrict__ Qbuf, int* __restrict__ active, double* __restrict__ diag,
    double tol, double skip_abs, int max_inner) {
  __shared__ JacLds lds;
  const int pidx = blockIdx.x;
  const int I = pairs[2 * pidx], J = pairs[2 * pidx + 1];
  const int tid = threadIdx.x;
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
    lds.s()[e / SB][e % SB] = v[it];
  }
  __syncthreads();
  pair_solve(lds, I, J, intra[pidx] != 0,
             JacSolve{nreal, Qbuf + (size_t)pidx * SB * SB, active + pidx, diag ? diag + (size_t)I * BS * BS : nullptr,
                      diag ? diag + (size_t)J * BS * BS : nullptr, tol, skip_abs, max_inner});
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

// One launch of the cross schedule: step s applied to A and C, and step
// s + 1's pair problems solved.
struct JacStep {
  const double* A;    // before the step
  double* Ao;         // after it (A itself where the step solves nothing ahead)
  double* C;
  int lda, nreal, npairs, npo, ntiles;
  const int* pairs;   // this step's pairs, rotations and active flags
  const double* q;
  const int* act;
  const int* pairs_n; // the next step's
  const int* intra_n;
  const int* where;   // per block: 2 x (its pair in this step) + which half
  double* qn;
  int* actn;
  const double* diag; // per block: its 32 x 32 diagonal block after this step
  double* diag_n;     // and after the next one
  double tol, skip_abs;
  int max_inner;
};

// Tile (P1 <= P2) of A: Ao(rows of P1, cols of P2) = Q1^T A Q2, and its
// mirror as the transpose, keeping A exactly symmetric.
__device__ __forceinline__ void step_tile_a(double* lds, const JacStep& a, int tile) {
  int P1, P2;
  tile_of(tile, a.npairs, a.npo, P1, P2);
  const bool a1 = a.act[P1] != 0, a2 = a.act[P2] != 0;
  const int lda = a.lda;
  if (!a1 && !a2 && a.A == a.Ao) return;
  // two 64 x 65 LDS tiles (66.5 KB) so two workgroups fit on a CU: the tile of
  // A, then Q1^T A, then the result; Q1, then Q2
  double(*At)[LDSW] = reinterpret_cast<double (*)[LDSW]>(lds);
  double(*Qs)[LDSW] = reinterpret_cast<double (*)[LDSW]>(lds + SB * LDSW);
  const int I1 = a.pairs[2 * P1], J1 = a.pairs[2 * P1 + 1];
  const int I2 = a.pairs[2 * P2], J2 = a.pairs[2 * P2 + 1];
  const int tid = threadIdx.x;
  const double* q1 = a.q + (size_t)P1 * SB * SB;
  const double* q2 = a.q + (size_t)P2 * SB * SB;
  // every global load of a stage is issued before the first LDS store, so a
  // thread waits for memory once per stage, not once per element; Q2 is
  // fetched into registers now and lands in LDS after the first product
  constexpr int PER = SB * SB / UPD_NT;  // element e = tid + 512 it: row tid % 64, column tid / 64 + 8 it
  double va[PER];
#pragma unroll
  for (int it = 0; it < PER; ++it) {
    const int e = tid + UPD_NT * it;
    va[it] = a.A[(size_t)gidx(I1, J1, e % SB) + (size_t)gidx(I2, J2, e / SB) * lda];
  }
  if (a1 || a2) {
    double vq[PER], vq2[PER];
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
  } else {
    // nothing rotates here: the tile moves to the other buffer as it is
#pragma unroll
    for (int it = 0; it < PER; ++it) {
      const int e = tid + UPD_NT * it;
      At[e % SB][e / SB] = va[it];
    }
  }
  __syncthreads();
  if (P1 == P2) {
    for (int e = tid; e < SB * SB; e += UPD_NT) {
      const int r = e % SB, c = e / SB;
      const double v = (r == c) ? At[r][c] : 0.5 * (At[r][c] + At[c][r]);
      a.Ao[(size_t)gidx(I1, J1, r) + (size_t)gidx(I2, J2, c) * lda] = v;
    }
    return;
  }
  for (int e = tid; e < SB * SB; e += UPD_NT) {
    const int r = e % SB, c = e / SB;
    a.Ao[(size_t)gidx(I1, J1, r) + (size_t)gidx(I2, J2, c) * lda] = At[r][c];
  }
  for (int e = tid; e < SB * SB; e += UPD_NT) {
    const int c = e % SB, r = e / SB;
    a.Ao[(size_t)gidx(I2, J2, c) + (size_t)gidx(I1, J1, r) * lda] = At[r][c];
  }
}

// C(64 rows from row0, cols of pair P) <- C(...) Q_P
__device__ __forceinline__ void step_tile_c(double* lds, const JacStep& a, int row0, int P) {
  if (!a.act[P]) return;
  double(*Ct)[LDSW] = reinterpret_cast<double (*)[LDSW]>(lds);
  double(*Qs)[LDSW] = reinterpret_cast<double (*)[LDSW]>(lds + SB * LDSW);
  const int I = a.pairs[2 * P], J = a.pairs[2 * P + 1];
  const double* q = a.q + (size_t)P * SB * SB;
  const int tid = threadIdx.x, ldc = a.lda;
  constexpr int PER = SB * SB / UPD_NT;
  double vc[PER], vq[PER];
#pragma unroll
  for (int it = 0; it < PER; ++it) {
    const int e = tid + UPD_NT * it;
    vc[it] = a.C[(size_t)(row0 + e % SB) + (size_t)gidx(I, J, e / SB) * ldc];
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
    a.C[(size_t)(row0 + r) + (size_t)gidx(I, J, c) * ldc] = Ct[r][c];
  }
}

// The 32x32 block (X, Y) of A after this step, Qx^T A Qy with the columns of
// X's and Y's pairs that belong to them, from A before it: 16x16 MFMA blocks,
// left in the first four waves (rows 16 (w / 2), columns 16 (w % 2) of the
// result).  A's operand is read from memory in the MFMA layout (16 lanes on
// consecutive rows); lds is free for the two halves of Q and A Qy.
__device__ __forceinline__ d4_t next_block(double* lds, const JacStep& a, int X, int Y) {
  constexpr int LH = BS + 1;
  double(*Tm)[LH] = reinterpret_cast<double (*)[LH]>(lds);
  double(*Qx)[LH] = reinterpret_cast<double (*)[LH]>(lds + SB * SB);
  double(*Qy)[LH] = reinterpret_cast<double (*)[LH]>(lds + SB * SB + SB * LH);
  const int wx = a.where[X], wy = a.where[Y];
  const int Px = wx >> 1, hx = wx & 1, Py = wy >> 1, hy = wy & 1;
  const int Ix = a.pairs[2 * Px], Jx = a.pairs[2 * Px + 1], Iy = a.pairs[2 * Py], Jy = a.pairs[2 * Py + 1];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int li = lane & 15, lk = lane >> 4;
  double av[16];
  {
    const size_t row = gidx(Ix, Jx, 16 * (w >> 1) + li);
#pragma unroll
    for (int i = 0; i < 16; ++i) av[i] = a.A[row + (size_t)gidx(Iy, Jy, 4 * i + lk) * a.lda];
  }
  constexpr int PER = SB * BS / CROSS_THREADS;
  double vx[PER], vy[PER];
  const double* qx = a.q + (size_t)Px * SB * SB + hx * SB * BS;
  const double* qy = a.q + (size_t)Py * SB * SB + hy * SB * BS;
  const bool ax = a.act[Px] != 0, ay = a.act[Py] != 0;
#pragma unroll
  for (int it = 0; it < PER; ++it) {
    const int e = tid + CROSS_THREADS * it, r = e % SB, c = e / SB;
    vx[it] = ax ? qx[e] : (r == BS * hx + c ? 1.0 : 0.0);
    vy[it] = ay ? qy[e] : (r == BS * hy + c ? 1.0 : 0.0);
  }
#pragma unroll
  for (int it = 0; it < PER; ++it) {
    const int e = tid + CROSS_THREADS * it;
    Qx[e % SB][e / SB] = vx[it];
    Qy[e % SB][e / SB] = vy[it];
  }
  __syncthreads();
  d4_t acc = d4_t{0.0, 0.0, 0.0, 0.0};
  const int cb = 16 * (w & 1);
#pragma unroll
  for (int i = 0; i < 16; ++i) acc = mfma16x16x4(av[i], Qy[4 * i + lk][cb + li], acc);
#pragma unroll
  for (int t = 0; t < 4; ++t) Tm[16 * (w >> 1) + lk + 4 * t][cb + li] = acc[t];
  __syncthreads();
  acc = d4_t{0.0, 0.0, 0.0, 0.0};
  if (w < 4) {
    const int rb = 16 * (w >> 1);
#pragma unroll
    for (int i = 0; i < 16; ++i) acc = mfma16x16x4(Qx[4 * i + lk][rb + li], Tm[4 * i + lk][cb + li], acc);
  }
  __syncthreads();
  return acc;
}

// Pair p of the next step: its 64x64 problem is put together from this
// step's rotations and A as it is before them, so the solve runs beside the
// updates of A and C that the same launch makes.  The two diagonal blocks are
// those the last solve of each block left; at the first step of a sweep they
// are formed from A as well, so that nothing drifts over the sweeps.
__device__ __forceinline__ void step_solve(JacLds& lds, const JacStep& a, int p) {
  const int I = a.pairs_n[2 * p], J = a.pairs_n[2 * p + 1];
  const bool do_intra = a.intra_n[p] != 0;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  double(*S)[SB] = lds.s();
  constexpr int PER = BS * BS / CROSS_THREADS;
  double vi[PER], vj[PER];
  if (!do_intra) {
#pragma unroll
    for (int it = 0; it < PER; ++it) {
      vi[it] = a.diag[(size_t)I * BS * BS + tid + CROSS_THREADS * it];
      vj[it] = a.diag[(size_t)J * BS * BS + tid + CROSS_THREADS * it];
    }
  }
  const d4_t lr = next_block(lds.m, a, I, J);
  const int r0 = 16 * (w >> 1) + (lane >> 4), c0 = 16 * (w & 1) + (lane & 15);
  if (do_intra) {
    const d4_t ll = next_block(lds.m, a, I, I);
    const d4_t rr = next_block(lds.m, a, J, J);
    if (w < 4) {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        S[r0 + 4 * t][c0] = ll[t];
        S[32 + r0 + 4 * t][32 + c0] = rr[t];
        S[32 + c0][r0 + 4 * t] = lr[t];
      }
    }
  } else {
#pragma unroll
    for (int it = 0; it < PER; ++it) {
      const int e = tid + CROSS_THREADS * it;
      S[e / BS][e % BS] = vi[it];
      S[32 + e / BS][32 + e % BS] = vj[it];
    }
  }
  if (w < 4) {
#pragma unroll
    for (int t = 0; t < 4; ++t) S[r0 + 4 * t][32 + c0] = lr[t];
  }
  __syncthreads();
  pair_solve(lds, I, J, do_intra,
             JacSolve{a.nreal, a.qn + (size_t)p * SB * SB, a.actn + p, a.diag_n + (size_t)I * BS * BS,
                      a.diag_n + (size_t)J * BS * BS, a.tol, a.skip_abs, a.max_inner});
}

// Workgroups [0, npairs) solve the next step's pairs, the next ntiles update
// A, the others C.  The solves are the longest and start first; they read A
// before the step while the update writes the other buffer, so nothing in
// the launch waits for anything else in it.
//
// Solving in a launch of its own left the chip to npairs workgroups for 22
// of a step's 37 us at 1020 orbitals (with the A update behind it, and the C
// update on a second stream, ordered by two events per step); this launch
// takes 24 us, of which the solve's 32 rounds are 12 (each a chain of about
// 940 cycles: LDS, the block, the next angle, a barrier) and putting its
// problem together 4.  At 3072 orbitals the updates set it (48 us).
__global__ __launch_bounds__(CROSS_THREADS, 4) void k_jac_step(JacStep a, int base) {
  static_assert(UPD_NT == CROSS_THREADS, "one workgroup size for every role");
  __shared__ JacLds lds;
  const int b = (int)blockIdx.x + base;
  if (b < a.npairs) {
    step_solve(lds, a, b);
  } else if (b < a.npairs + a.ntiles) {
    step_tile_a(lds.m, a, b - a.npairs);
  } else {
    const int c = b - a.npairs - a.ntiles, nrow = a.lda / SB;
    step_tile_c(lds.m, a, (c % nrow) * SB, c / nrow);
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

void jacobi_set_identity(hipStream_t s, int npad, double* C, int ldc) {
  hipLaunchKernelGGL(k_set_identity, dim3((npad + 255) / 256, npad), dim3(256), 0, s, npad, C, ldc);
  MHIP_LAUNCH_CHECK();
}

int jacobi_sweeps(hipStream_t s, JacobiPlan& plan, double*& A, double*& A2, double* C, double tol, int max_sweeps,
                  double* host_scal, double* dev_scal, int* sweeps_done) {
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
  const int ntiles = plan.npo * (plan.npo + 1) / 2 + npv * (npv + 1) / 2, nctiles = npairs * (plan.npad / SB);
  int slot = 0;  // of the step at hand in the two-step buffers
  auto qslot = [&](int k) { return plan.qbuf.as<double>() + (size_t)k * npairs * SB * SB; };
  auto aslot = [&](int k) { return plan.active.as<int>() + (size_t)k * npairs; };
  auto dslot = [&](int k) { return plan.diag.as<double>() + (size_t)k * plan.nb * BS * BS; };
  auto pairs_of = [&](int step) { return plan.pairs.as<int>() + (size_t)step * npairs * 2; };
  auto intra_of = [&](int step) { return plan.intra.as<int>() + (size_t)step * npairs; };
  auto solve = [&](int step, double skip_abs) {
    if (cross)
      hipLaunchKernelGGL(k_jac_solve_x, dim3(npairs), dim3(CROSS_THREADS), 0, s, A, lda, plan.n, pairs_of(step),
                         intra_of(step), qslot(slot), aslot(slot), ahead ? dslot(slot) : nullptr, inner_tol, skip_abs,
                         inner);
    else
      hipLaunchKernelGGL(k_jac_solve, dim3(npairs), dim3(SOLVE_THREADS), 0, s, A, lda, plan.n, pairs_of(step),
                         qslot(slot), aslot(slot), 1.0e-14, skip_abs, inner);
    MHIP_LAUNCH_CHECK();
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
      if (sweeps_done) *sweeps_done = done;
      return 1;
    }
    if (plan.timing && plan.ev.size() < (size_t)(6 * nsteps)) {
      for (auto e : plan.ev) (void)hipEventDestroy(e);
      plan.ev.assign(6 * nsteps, nullptr);
      for (auto& e : plan.ev) MHIP_CHECK(hipEventCreate(&e));
    }
    const bool timing = plan.timing && g_kernel_variant == 1;
    // part k of the step's launch between events 2 k and 2 k + 1
    auto mark = [&](int step, int k) {
      if (timing) MHIP_CHECK(hipEventRecord(plan.ev[6 * step + k], s));
    };
    // the first step's solve of a later sweep ran in the last launch of the
    // sweep before
    if (ahead && sw == 0) solve(0, skip_abs);
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
        const int next = (step + 1) % nsteps, first = ahead ? 0 : npairs, total = npairs + ntiles + nctiles;
        const JacStep a{A,          ahead ? A2 : A,  C,                lda,
                        plan.n,     npairs,          plan.npo,         ntiles,
                        pairs_of(step), qslot(slot), aslot(slot),      pairs_of(next),
                        intra_of(next), plan.where.as<int>() + (size_t)step * plan.nb, qslot(slot ^ 1), aslot(slot ^ 1),
                        dslot(slot), dslot(slot ^ 1), inner_tol,       skip_abs,
                        inner};
        auto launch = [&](int from, int to) {
          hipLaunchKernelGGL(k_jac_step, dim3(to - from), dim3(CROSS_THREADS), 0, s, a, from);
          MHIP_LAUNCH_CHECK();
        };
        if (!timing) {
          launch(first, total);
        } else {
          // the same work in a launch per part, for the parts' times
          if (ahead) {
            mark(step, 0);
            launch(0, npairs);
            mark(step, 1);
          }
          mark(step, 2);
          launch(npairs, npairs + ntiles);
          mark(step, 3);
          mark(step, 4);
          launch(npairs + ntiles, total);
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
