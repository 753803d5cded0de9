// Device code of the Fock row pass and of the packed storage, shared by the
// single-system kernels (k_fock.hip) and the batched SCF (k_batch.hip).
#pragma once
#include "common.h"
#include "k_fock.h"

namespace mhip {
namespace {

__constant__ int c_pa[10] = {0, 1, 1, 2, 2, 2, 3, 3, 3, 3};  // larger orbital of pair
__constant__ int c_pb[10] = {0, 0, 1, 0, 1, 2, 0, 1, 2, 3};  // smaller orbital of pair

__device__ __forceinline__ long long pk(long long r, long long c) {
  return r >= c ? r * (r + 1) / 2 + c : c * (c + 1) / 2 + r;
}

// Starting value of F(q) before G(P) is added.
__device__ __forceinline__ double finit(const FockArgs& a, long long q, bool diag) {
  switch (a.init_mode) {
    case kInitShift: {
      double v = a.h[q] + a.shift * a.pa[q] + 1.0e-16 * (double)(q + 1);
      if (diag) v -= a.shift;
      return v;
    }
    case kInitRandom:
      return a.h[q] + (((q + 1) & 1) ? -0.001 : 0.001);
    case kInitCopy:
      return a.fin[q];
    default:
      return a.h[q];
  }
}

// Row pass for atom i by NT threads, thread `lane` of them: a workgroup of
// 256, or one wave (a small molecule's atom has few partners).
template <int NT>
__device__ void fock_rows_body(const FockArgs& a, const int i, const int lane) {
  const int ni = a.sys.norb[i];
  const long long fi = a.sys.nf0[i];
  const double* __restrict__ P = a.p;
  const double* __restrict__ Pa = a.pa;
  // density of atom i with off-diagonal elements doubled
  double pi2[10];
  if (ni == 4) {
#pragma unroll
    for (int ab = 0; ab < 10; ++ab) {
      const int x = c_pa[ab], y = c_pb[ab];
      pi2[ab] = P[pk(fi + x, fi + y)] * (x == y ? 1.0 : 2.0);
    }
  } else {
    pi2[0] = P[pk(fi, fi)];
#pragma unroll
    for (int ab = 1; ab < 10; ++ab) pi2[ab] = 0.0;
  }
  double ji[10];
#pragma unroll
  for (int ab = 0; ab < 10; ++ab) ji[ab] = 0.0;

  const long long wrow = a.sys.woff[i];
  const int limi = (ni == 4) ? 10 : 1;
  const int nheavy = a.sys.nheavy_before[i];
  const int nlight = a.sys.nlight_before[i];

  // ---- heavy partners -------------------------------------------------------
  for (int t = lane; t < nheavy; t += NT) {
    const int j = a.sys.heavy[t];
    const long long fj = a.sys.nf0[j];
    double pj2[10];
#pragma unroll
    for (int cd = 0; cd < 10; ++cd) {
      const int x = c_pa[cd], y = c_pb[cd];
      pj2[cd] = P[pk(fj + x, fj + y)] * (x == y ? 1.0 : 2.0);
    }
    const double* __restrict__ wb = a.sys.w + wrow + (long long)limi * a.sys.wcum[j];
    double jj[10];
#pragma unroll
    for (int cd = 0; cd < 10; ++cd) jj[cd] = 0.0;
    const long long col = a.sys.ccol[j] + (long long)(i - j - 1) * 10;
    if (ni == 4) {
      double pa_ij[4][4], K[4][4];
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) {
          pa_ij[x][y] = Pa[pk(fi + x, fj + y)];
          K[x][y] = 0.0;
        }
#pragma unroll
      for (int ab = 0; ab < 10; ++ab) {
        const int x = c_pa[ab], y = c_pb[ab];
        double wr[10];
#pragma unroll
        for (int cd = 0; cd < 10; ++cd) wr[cd] = wb[ab * 10 + cd];
        double s = 0.0;
#pragma unroll
        for (int cd = 0; cd < 10; ++cd) {
          s = fma(wr[cd], pj2[cd], s);
          jj[cd] = fma(pi2[ab], wr[cd], jj[cd]);
          const int u = c_pa[cd], v = c_pb[cd];
          const double wv = wr[cd];
          K[x][u] = fma(pa_ij[y][v], wv, K[x][u]);
          if (x != y) K[y][u] = fma(pa_ij[x][v], wv, K[y][u]);
          if (u != v) K[x][v] = fma(pa_ij[y][u], wv, K[x][v]);
          if (x != y && u != v) K[y][v] = fma(pa_ij[x][u], wv, K[y][v]);
        }
        ji[ab] += s;
      }
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) {
          const long long q = pk(fi + x, fj + y);
          a.f[q] = finit(a, q, false) - K[x][y];
        }
    } else {
      // hydrogen i with heavy j: W block is the 10 pairs of atom j
      const double pii = pi2[0];
      double pa_ij[4], K[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int y = 0; y < 4; ++y) pa_ij[y] = Pa[pk(fi, fj + y)];
      double s = 0.0;
#pragma unroll
      for (int cd = 0; cd < 10; ++cd) {
        const double wv = wb[cd];
        s = fma(wv, pj2[cd], s);
        jj[cd] = pii * wv;
        const int u = c_pa[cd], v = c_pb[cd];
        K[u] = fma(pa_ij[v], wv, K[u]);
        if (u != v) K[v] = fma(pa_ij[u], wv, K[v]);
      }
      ji[0] += s;
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        const long long q = pk(fi, fj + y);
        a.f[q] = finit(a, q, false) - K[y];
      }
    }
#pragma unroll
    for (int cd = 0; cd < 10; ++cd) a.jcol[col + cd] = jj[cd];
  }

  // ---- hydrogen partners ----------------------------------------------------
  for (int t = lane; t < nlight; t += NT) {
    const int j = a.sys.light[t];
    const long long fj = a.sys.nf0[j];
    const double pjj = P[pk(fj, fj)];
    const double* __restrict__ wb = a.sys.w + wrow + (long long)limi * a.sys.wcum[j];
    const long long col = a.sys.ccol[j] + (long long)(i - j - 1);
    if (ni == 4) {
      double pa_ij[4], K[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int x = 0; x < 4; ++x) pa_ij[x] = Pa[pk(fi + x, fj)];
      double s = 0.0;
#pragma unroll
      for (int ab = 0; ab < 10; ++ab) {
        const double wv = wb[ab];
        ji[ab] = fma(wv, pjj, ji[ab]);
        s = fma(pi2[ab], wv, s);
        const int x = c_pa[ab], y = c_pb[ab];
        K[x] = fma(pa_ij[y], wv, K[x]);
        if (x != y) K[y] = fma(pa_ij[x], wv, K[y]);
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const long long q = pk(fi + x, fj);
        a.f[q] = finit(a, q, false) - K[x];
      }
      a.jcol[col] = s;
    } else {
      const double wv = wb[0];
      ji[0] = fma(wv, pjj, ji[0]);
      const long long q = pk(fi, fj);
      a.f[q] = finit(a, q, false) - Pa[q] * wv;
      a.jcol[col] = wv * pi2[0];
    }
  }

  // ---- reduce the Coulomb field on atom i over the workgroup -----------------
  if constexpr (NT == 64) {
    // one wave: lane exchange, fixed order
#pragma unroll
    for (int ab = 0; ab < 10; ++ab)
      for (int o = 32; o > 0; o >>= 1) ji[ab] += __shfl_xor(ji[ab], o);
    if (lane == 0)
      for (int ab = 0; ab < limi; ++ab) a.jrow[(long long)i * 10 + ab] = ji[ab];
  } else {
    __shared__ double red[10][NT];
#pragma unroll
    for (int ab = 0; ab < 10; ++ab) red[ab][lane] = ji[ab];
    __syncthreads();
    for (int w = NT / 2; w > 0; w >>= 1) {
      if (lane < w)
#pragma unroll
        for (int ab = 0; ab < 10; ++ab) red[ab][lane] += red[ab][lane + w];
      __syncthreads();
    }
    if (lane < limi) a.jrow[(long long)i * 10 + lane] = red[lane][0];
  }
}

}  // namespace
}  // namespace mhip
