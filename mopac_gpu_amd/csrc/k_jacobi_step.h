// Device code of the block-Jacobi steps: the 64x64 pair solve of the cross
// schedule and the tiles that apply a step to A and C.  Shared by the
// single-system eigensolver (k_eigen.hip) and the batched one
// (k_batch_eig.hip).
#pragma once
#include <utility>

#include "common.h"
#include "jacobi_rotation.h"
#include "mfma.h"

namespace mhip {
namespace {

constexpr int BS = 32;  // block width
constexpr int SB = 64;  // pair width
constexpr int LDSW = SB + 1;

__device__ __forceinline__ int gidx_dev(int pairI, int pairJ, int local) {
  return (local < BS) ? pairI * BS + local : pairJ * BS + (local - BS);
}

// The angles start in FP32: a problem with elements above this is solved as a
// power of two times one with elements up to 1, which has the same rotations.
// r^2 of a pair is at most (2 x 64 x 2^50)^2 in a 64 x 64 problem.
constexpr double kAngleRange = 0x1p50;
__device__ __forceinline__ bool out_of_range(double top) {
  return top > kAngleRange && top < __builtin_huge_val();
}

// What the levels of n orbitals are ordered by: a NaN is above all others, so
// that every level has a place of its own whatever a matrix holds, and the
// padding after them, whatever they are (ties go by index).
__device__ __forceinline__ double sort_key(double level, int i, int n) {
  return i < n && level == level ? level : __builtin_huge_val();
}

__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
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

// Returns whether another round follows (nr of them in all, a power of two).
template <int R>
__device__ __forceinline__ bool cross_round(double (*S)[SB], double2 (*rot)[32], double (*dgl)[SB], int k, int g,
                                            int nr, CrossRegs& v) {
  constexpr int SG = cross_sigma(R), b = R & 1;
  // rotation k of the next round acts on S[k][32 + (k ^ SGN)], which is in
  // this round's block of d = M
  constexpr int SGN = R < 31 ? cross_sigma(R + 1) : 0, M = R < 31 ? SG ^ SGN : 0;
  constexpr bool may_end = ((R + 1) & R) == 0;
  const bool more = R < 31 && (!may_end || nr != R + 1);
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
  const bool next_pair = more && v.d == M;
  lds_at<double>(S, lr) = next_pair ? 0.0 : npq;
  lds_at<double>(S, rl) = next_pair ? 0.0 : nqp;
  if (R < 31 && more) {
    if (g == mask_group(M)) {
      // lane k of the half-wave takes rotation k: where the block kept is
      // that of k ^ M, its S[q1][k2]
      const double other = lane_xor<M ? M : 1>(nqp);
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
  return more;
}

template <int... R>
__device__ __forceinline__ void cross_rounds(std::integer_sequence<int, R...>, double (*S)[SB], double2 (*rot)[32],
                                             double (*dgl)[SB], int k, int g, int nr, CrossRegs& v) {
  (void)(cross_round<R>(S, rot, dgl, k, g, nr, v) && ...);
}

// The pair solve.  An inner sweep is a level of 32 cross rounds, in which the
// 1024 index pairs across the two blocks are each rotated once, after, where
// intra[pair] is set, the levels that rotate the pairs inside the blocks: 16
// cross rounds between the 16-wide halves of both blocks at once, then 8, 4,
// 2 and 1 between ever smaller halves.  A level inside the blocks is the
// cross level with two index bits exchanged (the bit that tells the halves
// becomes the one that tells the blocks): S is addressed that way, where
// moving it there and back took 1.5 us more a level.  The sweep schedule sets intra
// once per sweep of the block's group, so every index pair of the matrix is
// rotated once per sweep, in about half the sequential rounds of a full
// 64-index inner sweep.
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
  double red_off[CROSS_THREADS / 64], red_dg[CROSS_THREADS / 64];
  __device__ double (*s())[SB] { return reinterpret_cast<double (*)[SB]>(m); }
  __device__ double (*q())[LDSW] { return reinterpret_cast<double (*)[LDSW]>(m + SB * SB); }
};

// What a pair solve reads besides its 64x64 problem and what it writes.
struct JacSolve {
  int nreal;
  double* q;      // 64 x 64 rotation, column-major (may be null)
  int* active;    // 1 where something rotated (may be null)
  double* di;     // the two 32 x 32 diagonal blocks after the solve (may be null)
  double* dj;
  double tol, skip_abs;
  int max_inner;
};

// Q's columns with index bits 5 and j exchanged.
__device__ __forceinline__ void exchange_q(CrossRegs& v, int k, int j) {
  const bool up = (k >> j) & 1;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const double x = __shfl_xor(up ? v.ql[i] : v.qr[i], 1 << j, 64);
    if (up) v.ql[i] = x;
    else v.qr[i] = x;
  }
}

// S by 2^e
__device__ __noinline__ void scale_problem(double (*S)[SB], int e) {
  for (int i = threadIdx.x; i < SB * SB; i += CROSS_THREADS) S[i / SB][i % SB] = ldexp(S[i / SB][i % SB], e);
  __syncthreads();
}

// Diagonalizes the problem in lds.s(): the upper right quadrant and the two
// diagonal ones, and the lower left one where do_intra asks for it.  Returns
// the inner sweeps it took (0: nothing rotated); with p.q null, Q is left in
// lds.q() and S in lds.s().  ANY: of any size; elsewhere the matrix is in the
// angles' range (a test here costs a step of the solver 0.7%).
template <bool ANY = false>
__device__ __forceinline__ int pair_solve(JacLds& lds, int I, int J, bool do_intra, const JacSolve& p) {
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
  int sweeps = 0, scale = 0;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // a round ends with the angles of the next, which wave 7 computes in three
  // of four rounds, 6, 5 or 0 in the others, while two waves share each SIMD:
  // 5% of an SCF at 24 to 1020 orbitals.  Update workgroups come after.
  if (wave == 7) __builtin_amdgcn_s_setprio(3);
  else if (wave >= 5) __builtin_amdgcn_s_setprio(2);
  else __builtin_amdgcn_s_setprio(1);
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
    if ((sw == 0 && off <= p.skip_abs) || off <= p.tol * fmax(dg, ANY ? ldexp(1.0, -scale) : 1.0)) break;
    if constexpr (ANY) {
      const double top = fmax(off, dg);
      if (sw == 0 && out_of_range(top)) {
        scale = __builtin_amdgcn_readfirstlane(ilogb(top) + 1);
        scale_problem(S, -scale);
      }
    }
    ++sweeps;
    for (int lv = do_intra ? 0 : 5; lv < 6; ++lv) {
      // nothing to rotate between a real index and the padding (a matrix that
      // is one pair problem)
      if (p.nreal <= (1 << lv)) continue;
      // index i of the level is pi(i) of S, bits 5 and lv exchanged: a level
      // inside the blocks only has other addresses, and Q's columns move.
      // pi(a ^ b) = pi(a) ^ pi(b), and the sigmas stay below bit lv.
      auto pi = [lv](int i) {
        const int x = ((i >> 5) ^ (i >> lv)) & 1;
        return i ^ (x << 5) ^ (x << lv);
      };
      const int up = 1 << lv, rk = pi(k), rd = pi(v.d), rg = pi(g), rq = rk ^ up, rk2 = rk ^ rd, rq2 = rq ^ rd;
      if (lv < 5) exchange_q(v, k, lv);
      const int nr = 1 << lv;
      v.lr = (rk * SB + rq2) * 8;
      v.rl = (rk2 * SB + rq) * 8;
      v.ll = S[rk][rk2];
      v.rr = S[rq][rq2];
      // angles of round 0 and the diagonals after it
      if (tid < 32) {
        const double app = S[rk][rk], aqq = S[rq][rq], apq = S[rk][rq];
        double c, sn, t;
        rotation_of(app, aqq, apq, c, sn, t);
        S[rk][rq] = 0.0;
        lds.rot[0][tid] = make_double2(c, sn);
        lds.dgl[0][tid] = app - t * apq;
        lds.dgl[0][32 + tid] = aqq + t * apq;
      }
      __syncthreads();
      cross_rounds(std::make_integer_sequence<int, 32>{}, S, lds.rot, lds.dgl, k, g, nr, v);
      cross_turn_q(v);
      // the moving columns back in order; sigma ends at the last basis mask
      const int SL = nr == 32 ? 16 : nr == 16 ? 15 : nr == 8 ? 7 : nr == 4 ? 2 : nr == 2 ? 1 : 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) v.qr[j] = __shfl(v.qr[j], (tid & 32) | (k ^ SL), 64);
      // S whole again: the diagonal blocks here, the upper right one is there
      // and gives the lower left one
      const int last = rq ^ SL, last2 = rq2 ^ SL;
      if (lv < 5 || do_intra) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int q = rq ^ rg ^ (j ? pi(16) : 0);
          S[q][rk] = S[rk][q];
        }
      }
      S[rk][rk2] = S[rk2][rk] = v.ll;
      S[last][last2] = S[last2][last] = v.rr;
      if (tid < SB) {
        const int r = pi(tid);
        S[r][r] = lds.dgl[(nr - 1) & 1][tid];
      }
      __syncthreads();
      if (lv < 5) exchange_q(v, k, lv);
    }
  }
  __builtin_amdgcn_s_setprio(0);
  if (ANY && scale) scale_problem(S, scale);
  if (p.di) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int e = (g + 16 * j) * BS + k;
      p.di[e] = S[g + 16 * j][k];
      p.dj[e] = S[32 + g + 16 * j][32 + k];
    }
  }
  if (tid == 0 && p.active) *p.active = sweeps > 0 ? 1 : 0;
  if (sweeps == 0) return 0;
  // Q to LDS, then out with consecutive lanes on consecutive rows
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    Q[4 * g + j][k] = v.ql[j];
    Q[4 * g + j][32 + k] = v.qr[j];
  }
  __syncthreads();
  if (p.q) {
#pragma unroll
    for (int e = tid; e < SB * SB; e += CROSS_THREADS) p.q[e] = Q[e % SB][e / SB];
  }
  return sweeps;
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

// The outcome of a sweep's stopping test, for a launch that does not wait for
// the host: max |off-diagonal| and max |diagonal| (stat, null where the host
// has decided) against tol.  done() also sets what a pair is left alone below.
struct SweepTest {
  const double* stat = nullptr;
  double tol = 0.0;
  bool first = false;  // of the sweeps: nothing is done out of the angles' range
  __device__ bool done(double& skip_abs) const {
    if (!stat) return false;
    const double thr = tol * fmax(1.0, stat[1]);
    skip_abs = 0.1 * thr;
    return stat[0] <= thr || (first && out_of_range(fmax(stat[0], stat[1])));
  }
};

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
  int crows = 0;      // > 0: C is two diagonal blocks, the first of crows 64-row tiles and npo pairs
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

// The pair solve on a matrix in memory.
__device__ __forceinline__ void solve_from_memory(JacLds& lds, const double* __restrict__ A, int lda, int I, int J,
                                                  bool do_intra, const JacSolve& p) {
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
  pair_solve(lds, I, J, do_intra, p);
}

}  // namespace
}  // namespace mhip
