// Pseudo-diagonalization (Stewart, Csaszar & Pulay 1982) as in
// src/matrix/diag.F90:16-163:
//   FMO = C_occ^T F C_virt (two GEMMs),
//   tiny = 0.05 max|FMO|,
//   for every (virtual i, occupied j) in that order whose |FMO| >= tiny and
//   |FMO/(e_j - e_i)| >= 1.5e-7, rotate columns j and i of C.
// FMO is not updated during the rotations, so every angle is known up front,
// and the rows of C are independent.  Within a row, rotation (i, j) needs the
// results of (i, j - 1) and (i - 1, j) only: the rotations pass through a
// chain of lanes, one per virtual, in the order of every element's updates.
#include <algorithm>

#include "common.h"
#include "k_pseudo.h"

namespace mhip {
namespace {

__global__ __launch_bounds__(256) void k_absmax_partial(long long len, const double* __restrict__ x,
                                                        double* __restrict__ part) {
  double m = 0.0;
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < len; i += (long long)gridDim.x * 256)
    m = fmax(m, fabs(x[i]));
  __shared__ double red[256];
  red[threadIdx.x] = m;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void k_absmax_final(int nb, const double* __restrict__ part,
                                                      double* __restrict__ out,
                                                      unsigned long long* __restrict__ count) {
  double m = 0.0;
  for (int i = threadIdx.x; i < nb; i += 256) m = fmax(m, part[i]);
  __shared__ double red[256];
  red[threadIdx.x] = m;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = 0.05 * red[0];
    *count = 0;
  }
}

// Rotation parameters for every (virtual, occupied) pair, exactly as
// diag.F90:130-153 computes them, in the order k_rotate reads them: entry
// [b][t][l] is virtual 64 b + l with occupied j0 + t - l of the nj from j0 on,
// kSkip where the pair is not rotated or there is none.
constexpr int kStep = 16;        // steps that k_rotate loads at once
constexpr int kFront = 64;       // room before a row in LDS
constexpr double kSkip = 2.0;    // no cosine
__global__ __launch_bounds__(256) void k_rot_params(int nocc, int j0, int nj, int nvirt, int steps,
                                                    const double* __restrict__ fmo,
                                                    const double* __restrict__ eig,
                                                    const double* __restrict__ tiny_dev, double bigeps,
                                                    double2* __restrict__ ab,
                                                    unsigned long long* __restrict__ count) {
  const long long len = (long long)((nvirt + 63) / 64) * steps * 64;
  const double tiny = tiny_dev[0];
  int rotated = 0;
  for (long long q = blockIdx.x * 256LL + threadIdx.x; q < len; q += (long long)gridDim.x * 256) {
    const int l = (int)(q & 63);
    const long long bt = q >> 6;
    const int v = (int)(bt / steps) * 64 + l, j = (int)(bt % steps) - l;
    double alpha = kSkip, beta = 0.0;
    if (v < nvirt && j >= 0 && j < nj) {
      const double c = fmo[(long long)v * nocc + j0 + j];
      if (!(fabs(c) < tiny)) {
        const double d = eig[j0 + j] - eig[nocc + v];
        if (!(fabs(c / d) < bigeps)) {
          const double e = (d >= 0.0 ? 1.0 : -1.0) * sqrt(4.0 * c * c + d * d);
          alpha = sqrt(0.5 * (1.0 + d / e));
          beta = -(c >= 0.0 ? 1.0 : -1.0) * sqrt(1.0 - alpha * alpha);
          ++rotated;
        }
      }
    }
    ab[q] = make_double2(alpha, beta);
  }
  for (int off = 32; off > 0; off >>= 1) rotated += __shfl_xor(rotated, off);
  __shared__ int part[4];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = rotated;
  __syncthreads();
  if (threadIdx.x == 0) {
    const int all = part[0] + part[1] + part[2] + part[3];
    if (all) atomicAdd(count, (unsigned long long)all);
  }
}

// lane l gets lane l - 1's value, lane 0 gets `first`
__device__ __forceinline__ double from_lane_below(double x, double first) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(first), __double2loint(x), 0x138, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(first), __double2hiint(x), 0x138, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

// All rotations of a row of C with the nocc occupied from column Co on, a row
// per wave.  64 virtuals at a time, one in
// each lane's register; at step t lane l rotates its virtual with occupied
// t - l, which comes from lane l - 1 as that left it, so the occupied
// coefficients stream from the row in LDS through the lanes and back.  The
// row has kStep-rounded room around it there: what enters lane 0 after the
// last occupied and leaves lane 63 before the first is not rotated.
// A step issues two lane shifts, four FP64 operations and the selects; its
// angles are one coalesced load, kStep steps ahead.  Several rows a wave
// would issue as much per row, on fewer of the chip's SIMDs.  The ordered
// list, a lane per row and one rotation after another with an LDS read and
// write each, took 434 us at 384 orbitals (256 occupied); this takes 37.
constexpr int kRotRows = 4;  // a workgroup's
__global__ __launch_bounds__(64 * kRotRows) void k_rotate(int n, int ldc, double* __restrict__ Co,
                                                          double* __restrict__ Cv, int nocc, int nvirt, int steps,
                                                          const double2* __restrict__ ab) {
  extern __shared__ double slab[];  // a row of kFront + steps per wave
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int len = kFront + steps;
  const int row0 = blockIdx.x * kRotRows, row = row0 + wave;
  for (int e = tid; e < kRotRows * nocc; e += 64 * kRotRows) {
    const int r = e % kRotRows, c = e / kRotRows;
    slab[r * len + kFront + c] = row0 + r < n ? Co[(size_t)(row0 + r) + (size_t)c * ldc] : 0.0;
  }
  __syncthreads();
  double* S = slab + wave * len;
  for (int v0 = 0; v0 < nvirt; v0 += 64) {
    double* col = Cv + (size_t)row + (size_t)(v0 + lane) * ldc;
    const bool have = v0 + lane < nvirt && row < n;
    double a = 0.0, b = have ? *col : 0.0;
    const double2* q = ab + (size_t)(v0 >> 6) * steps * 64 + lane;
    double2 next[kStep];
#pragma unroll
    for (int u = 0; u < kStep; ++u) next[u] = q[(size_t)u * 64];
    for (int t0 = 0; t0 < steps; t0 += kStep) {
      double2 rot[kStep];
#pragma unroll
      for (int u = 0; u < kStep; ++u) rot[u] = next[u];
      if (t0 + kStep < steps) {
#pragma unroll
        for (int u = 0; u < kStep; ++u) next[u] = q[(size_t)(t0 + kStep + u) * 64];
      }
      double x[kStep];
#pragma unroll
      for (int u = 0; u < kStep; ++u) x[u] = S[kFront + t0 + u];
#pragma unroll
      for (int u = 0; u < kStep; ++u) {
        const bool skip = rot[u].x == kSkip;
        a = from_lane_below(a, x[u]);
        const double na = rot[u].x * a + rot[u].y * b;
        const double nb = rot[u].x * b - rot[u].y * a;
        a = skip ? a : na;
        b = skip ? b : nb;
        x[u] = a;
      }
      // lane 63 is 63 steps behind lane 0, and behind this wave's reads
      if (lane == 63) {
#pragma unroll
        for (int u = 0; u < kStep; ++u) S[kFront - 63 + t0 + u] = x[u];
      }
    }
    if (have) *col = b;
    // every lane reads what lane 63 stored: not before this point, and not
    // from before it
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  __syncthreads();
  for (int e = tid; e < kRotRows * nocc; e += 64 * kRotRows) {
    const int r = e % kRotRows, c = e / kRotRows;
    if (row0 + r < n) Co[(size_t)(row0 + r) + (size_t)c * ldc] = slab[r * len + kFront + c];
  }
}

// Apply an ordered list of rotations of any two columns to `rows` consecutive
// rows of C held in LDS.
__global__ __launch_bounds__(64) void k_apply_rotations(int n, int ldc, double* __restrict__ C,
                                                        int rows, const long long* __restrict__ total,
                                                        const int2* __restrict__ cols,
                                                        const double2* __restrict__ rot) {
  extern __shared__ double slab[];  // rows x n, row-major
  const int row0 = blockIdx.x * rows;
  const int nr = min(rows, n - row0);
  for (int e = threadIdx.x; e < nr * n; e += 64) {
    const int r = e % nr, c = e / nr;
    slab[(size_t)r * n + c] = C[(size_t)(row0 + r) + (size_t)c * ldc];
  }
  __syncthreads();
  const long long nrot = *total;
  if (threadIdx.x < nr) {
    double* row = slab + (size_t)threadIdx.x * n;
    for (long long k = 0; k < nrot; ++k) {
      const int2 jc = cols[k];
      const double2 r = rot[k];
      const double a = row[jc.x], b = row[jc.y];
      row[jc.x] = r.x * a + r.y * b;
      row[jc.y] = r.x * b - r.y * a;
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < nr * n; e += 64) {
    const int r = e % nr, c = e / nr;
    C[(size_t)(row0 + r) + (size_t)c * ldc] = slab[(size_t)r * n + c];
  }
}

}  // namespace

// the first occupied enters lane 0 at step 0, the last leaves lane 63 at step
// nocc + 62
static int rot_steps(int nocc) { return (nocc + 63 + kStep - 1) / kStep * kStep; }
// The occupied levels go through in equal parts whose rows fit the LDS, each
// part past every virtual before the next: a virtual still meets them in
// order, and so does an occupied the virtuals.
constexpr int kMaxLds = 160 * 1024;
constexpr int kMaxPart = kMaxLds / (int)sizeof(double) / kRotRows - kFront - 63 - kStep;
static int rot_part(int nocc) {
  const int parts = (nocc + kMaxPart - 1) / kMaxPart;
  return (nocc + parts - 1) / parts;
}

void PseudoWork::ensure(int n, int nocc, int ld) {
  const long long nvirt = n - nocc;
  const long long len = (long long)nocc * nvirt;
  fd.ensure(sizeof(double) * (size_t)ld * ld);
  wv.ensure(sizeof(double) * (size_t)ld * std::max<long long>(nvirt, 1));
  fmo.ensure(sizeof(double) * std::max<long long>(len, 1));
  ab.ensure(sizeof(double2) * ((nvirt + 63) / 64) * 64 * rot_steps(rot_part(nocc)));
  part.ensure(sizeof(double) * 1032);
}

void PseudoWork::release() {
  for (DevBuf* b : {&fd, &wv, &fmo, &ab, &part}) b->release();
}

void pseudo_diag_device(hipStream_t s, PseudoWork& w, int n, int ld, const double* fpacked,
                        double* C, int nocc, const double* eig, long long* nrot_out) {
  const int nvirt = n - nocc;
  if (nvirt <= 0 || nocc <= 0) {
    if (nrot_out) *nrot_out = 0;
    return;
  }
  w.ensure(n, nocc, ld);
  unpack_sym(s, n, fpacked, w.fd.as<double>(), ld, n, 0.0);
  // Wv = F C_virt (n x nvirt), FMO = C_occ^T Wv (nocc x nvirt)
  gemm(s, 'N', 'N', n, nvirt, n, 1.0, w.fd.as<double>(), ld, C + (size_t)nocc * ld, ld, 0.0,
       w.wv.as<double>(), ld);
  gemm(s, 'T', 'N', nocc, nvirt, n, 1.0, C, ld, w.wv.as<double>(), ld, 0.0, w.fmo.as<double>(), nocc);
  const long long len = (long long)nocc * nvirt;
  const int nb = (int)std::min<long long>(1024, (len + 255) / 256);
  hipLaunchKernelGGL(k_absmax_partial, dim3(nb), dim3(256), 0, s, len, w.fmo.as<double>(),
                     w.part.as<double>());
  MHIP_LAUNCH_CHECK();
  unsigned long long* count = reinterpret_cast<unsigned long long*>(w.part.as<double>() + 1024);
  hipLaunchKernelGGL(k_absmax_final, dim3(1), dim3(256), 0, s, nb, w.part.as<double>(),
                     w.part.as<double>() + 1023, count);
  MHIP_LAUNCH_CHECK();
  MHIP_CHECK(hipFuncSetAttribute((const void*)k_rotate, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds));
  const int part = rot_part(nocc);
  for (int j0 = 0; j0 < nocc; j0 += part) {
    const int nj = std::min(part, nocc - j0), steps = rot_steps(nj);
    const long long entries = (long long)((nvirt + 63) / 64) * 64 * steps;
    hipLaunchKernelGGL(k_rot_params, dim3((int)std::min<long long>(512, (entries + 255) / 256)), dim3(256), 0, s, nocc,
                       j0, nj, nvirt, steps, w.fmo.as<double>(), eig, w.part.as<double>() + 1023, 1.5e-7,
                       w.ab.as<double2>(), count);
    MHIP_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_rotate, dim3((n + kRotRows - 1) / kRotRows), dim3(64 * kRotRows),
                       sizeof(double) * kRotRows * (kFront + steps), s, n, ld, C + (size_t)j0 * ld,
                       C + (size_t)nocc * ld, nj, nvirt, steps, w.ab.as<double2>());
    MHIP_LAUNCH_CHECK();
  }
  if (nrot_out) {
    MHIP_CHECK(hipMemcpyAsync(nrot_out, count, sizeof(long long), hipMemcpyDeviceToHost, s));
    MHIP_CHECK(hipStreamSynchronize(s));
  }
}

void apply_rotation_list(hipStream_t s, int n, int ld, double* C, const long long* nrot_dev,
                         const int2* cols, const double2* rot) {
  const int rows = std::max(1, std::min(64, 19456 / n));
  const size_t lds = sizeof(double) * (size_t)rows * n;
  MHIP_CHECK(hipFuncSetAttribute((const void*)k_apply_rotations,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
  hipLaunchKernelGGL(k_apply_rotations, dim3((n + rows - 1) / rows), dim3(64), lds, s, n, ld, C,
                     rows, nrot_dev, cols, rot);
  MHIP_LAUNCH_CHECK();
}

}  // namespace mhip
