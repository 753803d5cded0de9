// Batched block-Jacobi eigensolver: the diagonalization of many molecules of
// 65 to 256 orbitals at once, each spread over several workgroups.
//
// The steps are those of the single-system solver (k_jacobi_step.h): one
// launch applies step s to every molecule's A and C and solves step s + 1's
// pair problems.  Molecules of one padded size (128, 192, 256) share a
// schedule; those whose matrix has converged drop out of the launches by a
// flag, tested once per sweep.  The warm start A = C^T F C, the density and
// the final ordering are batched the same way.
//
// In one workgroup per molecule, A packed in its LDS, a 180-orbital
// eigensolve took 5 ms (179 rounds a sweep, each two barriers over all of A,
// and C turned from a log of the rotations), so 50 such molecules took as
// long as 250 would have; here a step of all molecules is a launch, 55 us on
// average with 150 of them (a sweep is 3, 5 or 7 steps).
#include <algorithm>
#include <vector>

#include "common.h"
#include "k_batch.h"
#include "k_eigen.h"
#include "k_jacobi_step.h"
#include "mfma.h"

namespace mhip {
namespace {

constexpr int kGroups = 3;    // padded sizes 128, 192, 256
constexpr int kMaxSweeps = kEigSweeps;

struct BjMol {
  int mol;         // index in the batch
  int n, nocc, npad;
  double* A[2];    // the matrix before and after a step, in turn
  double* C;       // working eigenvectors
  double* Cs;      // ordered eigenvectors of the last solve (the warm start)
  double* T;       // F C: A[1], before the first step writes it
  double* q;       // rotations, flags and diagonal blocks of two steps
  int* act;
  double* diag;
  double *f, *p, *eig;
};

struct BjState {
  int run;         // still sweeping
  int did;         // this call diagonalizes the molecule
  int cur;         // which A holds the result
  int sweeps;
  int stuck;       // out of sweeps
  int scale;       // A is the matrix times 2^-scale
  double skip;     // pairs this diagonal are left alone
  unsigned long long rot;
};

struct BjGroup {
  int npad, nb, npairs, nsteps, ntiles, nctiles;
  int first, count;  // its molecules in the table
  const int *pairs, *intra, *where;
};

struct BjLaunch {
  const BjMol* mol;
  BjState* st;
  BjGroup g[kGroups];
  int on[kGroups];    // the group takes part in this launch
  int par[kGroups];   // which A it reads
  int step;
  double tol;
};

// Workgroup b of a launch with per(g) workgroups for each molecule of group g:
// the group, molecule and workgroup within it; false past the last
template <class P>
__device__ __forceinline__ bool locate(const BjLaunch& a, int& b, int& g, int& m, const P& per) {
  for (g = 0; g < kGroups; ++g) {
    if (!a.on[g]) continue;
    const int len = a.g[g].count * per(a.g[g]);
    if (b < len) {
      m = a.g[g].first + b / per(a.g[g]);
      b %= per(a.g[g]);
      return true;
    }
    b -= len;
  }
  return false;
}

// F(i,i) += i * 1e-10 in place, as eigenvectors_LAPACK does, and the solve's
// starting state; counts[0] = molecules that are not done
__global__ __launch_bounds__(256) void k_bj_begin(const BjMol* __restrict__ mols, BjState* __restrict__ st,
                                                  const int* __restrict__ do_eig, const BatchState* __restrict__ bst,
                                                  int first, int* __restrict__ counts) {
  const int i = first + blockIdx.x;
  const BjMol& M = mols[i];
  const bool go = do_eig[M.mol] != 0;
  if (go)
    for (int k = threadIdx.x; k < M.n; k += 256) M.f[(size_t)k * (k + 1) / 2 + k] += (double)(k + 1) * 1.0e-10;
  if (threadIdx.x == 0) {
    st[i] = BjState{go ? 1 : 0, go ? 1 : 0, 0, 0, 0, 0, 0.0, 0ull};
    if (!bst[M.mol].done) atomicAdd(counts, 1);
  }
}

__global__ void k_bj_zero(int n, int* __restrict__ p) {
  if ((int)threadIdx.x < n) p[threadIdx.x] = 0;
}

// One 64x64 tile of X Y over nk chunks of 64: load(kc, it) gives this
// thread's element it of both chunks and where it goes
template <class L>
__device__ __forceinline__ void mm_tile(double* lds, int nk, const L& load, d4_t acc[2]) {
  double(*Xs)[LDSW] = reinterpret_cast<double (*)[LDSW]>(lds);
  double(*Ys)[LDSW] = reinterpret_cast<double (*)[LDSW]>(lds + SB * LDSW);
  acc[0] = acc[1] = d4_t{0.0, 0.0, 0.0, 0.0};
  for (int kc = 0; kc < nk; ++kc) {
    constexpr int PER = SB * SB / UPD_NT;
    double x[PER], y[PER];
#pragma unroll
    for (int it = 0; it < PER; ++it) load(kc, (int)threadIdx.x + UPD_NT * it, x[it], y[it]);
    if (kc) __syncthreads();
#pragma unroll
    for (int it = 0; it < PER; ++it) load.put((int)threadIdx.x + UPD_NT * it, x[it], y[it], Xs, Ys);
    __syncthreads();
    mfma_tile64_w8([&](int r, int k) { return Xs[r][k]; }, [&](int k, int c) { return Ys[k][c]; }, SB, acc);
  }
}

__device__ __forceinline__ double f_padded(const BjMol& M, int r, int c) {
  if (r < M.n && c < M.n) {
    const int a = max(r, c), b = min(r, c);
    return M.f[(size_t)a * (a + 1) / 2 + b];
  }
  return r == c ? 1.0e4 + r : 0.0;
}

// T = F C and the working copy of C, tile by tile; from a molecule without
// eigenvectors A = F and C = I instead
struct LoadFC {
  const BjMol& M;
  int r0, c0;
  __device__ void operator()(int kc, int e, double& x, double& y) const {
    x = f_padded(M, r0 + e % SB, 64 * kc + e / SB);
    y = M.Cs[(size_t)(64 * kc + e % SB) + (size_t)(c0 + e / SB) * M.npad];
  }
  __device__ void put(int e, double x, double y, double (*X)[LDSW], double (*Y)[LDSW]) const {
    X[e % SB][e / SB] = x;
    Y[e % SB][e / SB] = y;
  }
};
__global__ __launch_bounds__(UPD_NT) void k_bj_fc(BjLaunch a, const BatchState* __restrict__ bst) {
  __shared__ double lds[2 * SB * LDSW];
  int b = blockIdx.x, g, m;
  if (!locate(a, b, g, m, [](const BjGroup& q) { return (q.npad / SB) * (q.npad / SB); })) return;
  if (!a.st[m].did) return;
  const BjMol& M = a.mol[m];
  const int nt = M.npad / SB, r0 = SB * (b % nt), c0 = SB * (b / nt), tid = threadIdx.x;
  if (!bst[M.mol].have_c) {
    for (int e = tid; e < SB * SB; e += UPD_NT) {
      const int r = r0 + e % SB, c = c0 + e / SB;
      M.A[0][(size_t)r + (size_t)c * M.npad] = f_padded(M, r, c);
      M.C[(size_t)r + (size_t)c * M.npad] = r == c ? 1.0 : 0.0;
    }
    return;
  }
  d4_t acc[2];
  mm_tile(lds, nt, LoadFC{M, r0, c0}, acc);
  mfma_tile64_w8_store(acc, [&](int r, int c, double v) { M.T[(size_t)(r0 + r) + (size_t)(c0 + c) * M.npad] = v; });
  for (int e = tid; e < SB * SB; e += UPD_NT) {
    const size_t at = (size_t)(r0 + e % SB) + (size_t)(c0 + e / SB) * M.npad;
    M.C[at] = M.Cs[at];
  }
}

// A = C^T T on the tiles on and above the diagonal, mirrored
struct LoadCT {
  const BjMol& M;
  int r0, c0;
  __device__ void operator()(int kc, int e, double& x, double& y) const {
    x = M.Cs[(size_t)(64 * kc + e % SB) + (size_t)(r0 + e / SB) * M.npad];
    y = M.T[(size_t)(64 * kc + e % SB) + (size_t)(c0 + e / SB) * M.npad];
  }
  __device__ void put(int e, double x, double y, double (*X)[LDSW], double (*Y)[LDSW]) const {
    X[e / SB][e % SB] = x;
    Y[e % SB][e / SB] = y;
  }
};
__global__ __launch_bounds__(UPD_NT) void k_bj_ctf(BjLaunch a, const BatchState* __restrict__ bst) {
  __shared__ double lds[2 * SB * LDSW];
  int b = blockIdx.x, g, m;
  if (!locate(a, b, g, m, [](const BjGroup& q) { return (q.npad / SB) * (q.npad / SB + 1) / 2; })) return;
  const BjMol& M = a.mol[m];
  if (!a.st[m].did || !bst[M.mol].have_c) return;
  int ti, tj;
  tri_of(b, ti, tj);
  const int r0 = SB * ti, c0 = SB * tj;
  d4_t acc[2];
  mm_tile(lds, M.npad / SB, LoadCT{M, r0, c0}, acc);
  double(*O)[LDSW] = reinterpret_cast<double (*)[LDSW]>(lds);
  __syncthreads();
  mfma_tile64_w8_store(acc, [&](int r, int c, double v) { O[r][c] = v; });
  __syncthreads();
  double* A = M.A[0];
  for (int e = threadIdx.x; e < SB * SB; e += UPD_NT) {
    const int r = e % SB, c = e / SB;
    const double v = ti == tj && r != c ? 0.5 * (O[r][c] + O[c][r]) : O[r][c];
    A[(size_t)(r0 + r) + (size_t)(c0 + c) * M.npad] = v;
    if (ti != tj) A[(size_t)(c0 + r) + (size_t)(r0 + c) * M.npad] = O[c][r];
  }
}

// max|offdiag| <= tol max(1, max|diag|) over the molecule's n x n block: stop,
// or go on with the pairs that are not yet a tenth of that.  A matrix out of
// the angles' range is scaled before its first sweep, its largest element to
// 2^10.
__global__ __launch_bounds__(1024) void k_bj_test(BjLaunch a, int sweep, int last, int* __restrict__ count) {
  int b = blockIdx.x, g, m;
  if (!locate(a, b, g, m, [](const BjGroup&) { return 1; })) return;
  if (!a.st[m].run) return;
  const BjMol& M = a.mol[m];
  double* A = M.A[a.par[g]];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  double off = 0.0, dg = 0.0;
  for (int c = w; c < M.n; c += 16)
    for (int r = lane; r <= c; r += 64) {
      const double v = fabs(A[(size_t)r + (size_t)c * M.npad]);
      if (r == c) dg = fmax(dg, v);
      else off = fmax(off, v);
    }
  __shared__ double ro[16], rd[16];
  off = wave_max(off);
  dg = wave_max(dg);
  if (lane == 0) {
    ro[w] = off;
    rd[w] = dg;
  }
  __syncthreads();
  for (int i = 0; i < 16; ++i) {
    off = fmax(off, ro[i]);
    dg = fmax(dg, rd[i]);
  }
  BjState& s = a.st[m];
  if (const double top = fmax(off, dg); sweep == 0 && out_of_range(top)) {
    const int e = ilogb(top) - 10;
    for (int i = tid; i < M.npad * M.npad; i += 1024) A[i] = ldexp(A[i], -e);
    off = ldexp(off, -e);
    dg = ldexp(dg, -e);
    if (tid == 0) s.scale = e;
  }
  if (tid != 0) return;
  const double thr = a.tol * fmax(1.0, dg);
  s.cur = a.par[g];
  if (off <= thr || last) {
    s.run = 0;
    s.stuck = !(off <= thr);
  } else {
    s.skip = 0.1 * thr;
    s.sweeps += 1;
    atomicAdd(count, 1);
  }
}

__device__ __forceinline__ JacStep step_args(const BjLaunch& a, const BjGroup& G, int par, int m) {
  const BjMol& M = a.mol[m];
  const int next = (a.step + 1) % G.nsteps;
  const size_t qs = (size_t)G.npairs * SB * SB, ds = (size_t)G.nb * BS * BS;
  return JacStep{M.A[par], M.A[par ^ 1], M.C, G.npad, M.n, G.npairs, G.npairs, G.ntiles,
                 G.pairs + (size_t)a.step * G.npairs * 2, M.q + par * qs, M.act + par * G.npairs,
                 G.pairs + (size_t)next * G.npairs * 2, G.intra + (size_t)next * G.npairs,
                 G.where + (size_t)a.step * G.nb, M.q + (par ^ 1) * qs, M.act + (par ^ 1) * G.npairs,
                 M.diag + par * ds, M.diag + (par ^ 1) * ds, 1.0e-14, a.st[m].skip, 1};
}

__device__ __forceinline__ void count_rotations(BjState& s, int active, bool intra) {
  if (threadIdx.x == 0 && active) atomicAdd(&s.rot, (unsigned long long)(1024 + (intra ? 992 : 0)));
}

// the first step's pair problems of a solve, from A[0]
__global__ __launch_bounds__(CROSS_THREADS, 4) void k_bj_first(BjLaunch a) {
  __shared__ JacLds lds;
  int b = blockIdx.x, g, m;
  if (!locate(a, b, g, m, [](const BjGroup& q) { return q.npairs; })) return;
  if (!a.st[m].run) return;
  const BjMol& M = a.mol[m];
  const BjGroup& G = a.g[g];
  const int I = G.pairs[2 * b], J = G.pairs[2 * b + 1];
  const bool intra = G.intra[b] != 0;
  solve_from_memory(lds, M.A[0], G.npad, I, J, intra,
                    JacSolve{M.n, M.q + (size_t)b * SB * SB, M.act + b, M.diag + (size_t)I * BS * BS,
                             M.diag + (size_t)J * BS * BS, 1.0e-14, a.st[m].skip, 1});
  if (threadIdx.x == 0) count_rotations(a.st[m], M.act[b], intra);
}

// One step of every running molecule: the next step's solves of all of them
// first (the longest), then the tiles of A, then those of C.
__global__ __launch_bounds__(CROSS_THREADS, 4) void k_bj_step(BjLaunch a) {
  __shared__ JacLds lds;
  int b = blockIdx.x, g, m;
  if (locate(a, b, g, m, [](const BjGroup& q) { return q.npairs; })) {
    if (!a.st[m].run) return;
    const JacStep s = step_args(a, a.g[g], a.par[g], m);
    step_solve(lds, s, b);
    if (threadIdx.x == 0) count_rotations(a.st[m], s.actn[b], s.intra_n[b] != 0);
  } else if (locate(a, b, g, m, [](const BjGroup& q) { return q.ntiles; })) {
    if (!a.st[m].run) return;
    step_tile_a(lds.m, step_args(a, a.g[g], a.par[g], m), b);
  } else if (locate(a, b, g, m, [](const BjGroup& q) { return q.nctiles; })) {
    if (!a.st[m].run) return;
    const int nrow = a.g[g].npad / SB;
    step_tile_c(lds.m, step_args(a, a.g[g], a.par[g], m), (b % nrow) * SB, b / nrow);
  }
}

// levels and eigenvectors in ascending order (ties by index), and the counts
__global__ __launch_bounds__(512) void k_bj_order(BjLaunch a, BatchState* __restrict__ bst) {
  __shared__ double d[kMaxBatchN];
  __shared__ int from[kMaxBatchN];
  int b = blockIdx.x, g, m;
  if (!locate(a, b, g, m, [](const BjGroup&) { return 1; })) return;
  const BjState& s = a.st[m];
  if (!s.did) return;
  const BjMol& M = a.mol[m];
  const int np = M.npad, tid = threadIdx.x;
  const double* A = M.A[s.cur];
  const double level = tid < np ? ldexp(A[(size_t)tid + (size_t)tid * np], s.scale) : 0.0;
  const double key = sort_key(level, tid, M.n);
  if (tid < np) d[tid] = key;
  __syncthreads();
  if (tid < np) {
    int rank = 0;
    for (int j = 0; j < np; ++j) rank += (d[j] < key) || (d[j] == key && j < tid);
    from[rank] = tid;
    if (rank < M.n) M.eig[rank] = level;
  }
  __syncthreads();
  for (int e = tid; e < np * np; e += 512) M.Cs[e] = M.C[(size_t)(e % np) + (size_t)from[e / np] * np];
  if (tid == 0) {
    BatchState& t = bst[M.mol];
    const double dn = M.n, tn = 0.5 * dn * (dn + 1.0);
    t.eig_rot += (long long)s.rot;
    t.eig_flops += 12.0 * dn * (double)s.rot + (t.have_c ? 2.0 * dn * dn * dn + 2.0 * dn * tn : 0.0) + 2.0 * tn * M.nocc;
    t.sweeps += s.sweeps;
    t.last_sweeps = s.sweeps;
    t.stuck |= s.stuck;
    t.ndiag += 1;
    t.have_c = 1;
  }
}

// P = 2 C_occ C_occ^T, packed
struct LoadCC {
  const BjMol& M;
  int r0, c0;
  __device__ void operator()(int kc, int e, double& x, double& y) const {
    const int k = 64 * kc + e / SB;
    const bool in = k < M.nocc;
    x = in ? M.Cs[(size_t)(r0 + e % SB) + (size_t)k * M.npad] : 0.0;
    y = in ? M.Cs[(size_t)(c0 + e % SB) + (size_t)k * M.npad] : 0.0;
  }
  __device__ void put(int e, double x, double y, double (*X)[LDSW], double (*Y)[LDSW]) const {
    X[e % SB][e / SB] = x;
    Y[e / SB][e % SB] = y;
  }
};
__global__ __launch_bounds__(UPD_NT) void k_bj_density(BjLaunch a) {
  __shared__ double lds[2 * SB * LDSW];
  int b = blockIdx.x, g, m;
  if (!locate(a, b, g, m, [](const BjGroup& q) { return (q.npad / SB) * (q.npad / SB + 1) / 2; })) return;
  if (!a.st[m].did) return;
  const BjMol& M = a.mol[m];
  int tj, ti;
  tri_of(b, tj, ti);
  d4_t acc[2];
  mm_tile(lds, (M.nocc + SB - 1) / SB, LoadCC{M, SB * ti, SB * tj}, acc);
  mfma_tile64_w8_store(acc, [&](int r, int c, double v) {
    const int i = SB * ti + r, j = SB * tj + c;
    if (i < M.n && j <= i) M.p[(size_t)i * (i + 1) / 2 + j] = 2.0 * v;
  });
}

}  // namespace

struct BatchJacobi {
  JacobiPlan plan[kGroups];
  BjGroup g[kGroups] = {};
  DevBuf mols, st, dense, q, act, diag, counts;
  int* host = nullptr;  // pinned copy of counts
  hipEvent_t tested = nullptr;
  int n = 0;
};

BatchJacobi* bj_create(const std::vector<BatchMol>& mol, const std::vector<int>& which) {
  auto* j = new BatchJacobi();
  std::vector<BjMol> t;
  size_t dense = 0, q = 0, act = 0, diag = 0;
  for (int g = 0; g < kGroups; ++g) {
    BjGroup& G = j->g[g];
    G.npad = 128 + 64 * g;
    G.first = (int)t.size();
    for (int m : which) {
      const BatchMol& b = mol[m];
      if ((b.n + SB - 1) / SB * SB != G.npad) continue;
      BjMol x{};
      x.mol = m;
      x.n = b.n;
      x.nocc = b.nocc;
      x.npad = G.npad;
      x.f = b.f;
      x.p = b.p;
      x.eig = b.eig;
      t.push_back(x);
    }
    G.count = (int)t.size() - G.first;
    if (G.count == 0) continue;
    JacobiPlan& p = j->plan[g];
    p.build(G.npad);
    G.nb = p.nb;
    G.npairs = p.npairs;
    G.nsteps = p.nsteps;
    G.ntiles = p.npairs * (p.npairs + 1) / 2;
    G.nctiles = p.npairs * (G.npad / SB);
    G.pairs = p.pairs.as<int>();
    G.intra = p.intra.as<int>();
    G.where = p.where.as<int>();
    dense += (size_t)G.count * 4 * G.npad * G.npad;
    q += (size_t)G.count * 2 * G.npairs * SB * SB;
    act += (size_t)G.count * 2 * G.npairs;
    diag += (size_t)G.count * 2 * G.nb * BS * BS;
  }
  j->n = (int)t.size();
  MHIP_REQUIRE(j->n == (int)which.size(), "batched eigensolver: molecule outside 65 to 256 orbitals");
  j->dense.ensure(sizeof(double) * std::max<size_t>(dense, 1));
  j->q.ensure(sizeof(double) * std::max<size_t>(q, 1));
  j->act.ensure(sizeof(int) * std::max<size_t>(act, 1));
  j->diag.ensure(sizeof(double) * std::max<size_t>(diag, 1));
  double *d = j->dense.as<double>(), *pq = j->q.as<double>(), *pd = j->diag.as<double>();
  int* pa = j->act.as<int>();
  for (int g = 0; g < kGroups; ++g)
    for (int i = j->g[g].first; i < j->g[g].first + j->g[g].count; ++i) {
      BjMol& x = t[i];
      const size_t sz = (size_t)x.npad * x.npad;
      for (double** b : {&x.A[0], &x.A[1], &x.C, &x.Cs}) {
        *b = d;
        d += sz;
      }
      x.T = x.A[1];
      x.q = pq;
      pq += (size_t)2 * j->g[g].npairs * SB * SB;
      x.act = pa;
      pa += 2 * j->g[g].npairs;
      x.diag = pd;
      pd += (size_t)2 * j->g[g].nb * BS * BS;
    }
  j->mols.ensure(sizeof(BjMol) * std::max<size_t>(t.size(), 1));
  j->st.ensure(sizeof(BjState) * std::max<size_t>(t.size(), 1));
  j->counts.ensure(sizeof(int) * (kMaxSweeps + 2));
  MHIP_CHECK(hipHostMalloc((void**)&j->host, sizeof(int) * (kMaxSweeps + 2), hipHostMallocDefault));
  MHIP_CHECK(hipEventCreateWithFlags(&j->tested, hipEventDisableTiming));
  if (!t.empty()) MHIP_CHECK(hipMemcpy(j->mols.ptr, t.data(), sizeof(BjMol) * t.size(), hipMemcpyHostToDevice));
  return j;
}

void bj_destroy(BatchJacobi* j) {
  if (!j) return;
  for (auto& p : j->plan) p.release();
  for (DevBuf* b : {&j->mols, &j->st, &j->dense, &j->q, &j->act, &j->diag, &j->counts}) b->release();
  if (j->host) (void)hipHostFree(j->host);
  if (j->tested) (void)hipEventDestroy(j->tested);
  delete j;
}

int bj_solve(BatchJacobi* j, hipStream_t s, BatchState* bst, const int* do_eig, double tol, int max_sweeps, int lo,
             int hi) {
  BjLaunch a{};
  a.mol = j->mols.as<BjMol>();
  a.st = j->st.as<BjState>();
  a.tol = tol;
  int nmol = 0, nsteps = 0;
  for (int g = 0; g < kGroups; ++g) {
    a.g[g] = j->g[g];
    a.on[g] = j->g[g].count > 0 && j->g[g].npad >= lo && j->g[g].npad <= hi;
    if (!a.on[g]) continue;
    nmol += j->g[g].count;
    nsteps = std::max(nsteps, j->g[g].nsteps);
  }
  if (nmol == 0) return 0;
  auto total = [&](auto per) {
    int n = 0;
    for (int g = 0; g < kGroups; ++g)
      if (a.on[g]) n += a.g[g].count * per(a.g[g]);
    return n;
  };
  auto tiles = [](const BjGroup& g) { return (g.npad / SB) * (g.npad / SB + 1) / 2; };
  int* counts = j->counts.as<int>();
  hipLaunchKernelGGL(k_bj_zero, dim3(1), dim3(64), 0, s, kMaxSweeps + 2, counts);
  MHIP_LAUNCH_CHECK();
  for (int g = 0; g < kGroups; ++g) {
    if (!a.on[g]) continue;
    hipLaunchKernelGGL(k_bj_begin, dim3(a.g[g].count), dim3(256), 0, s, a.mol, a.st, do_eig, bst, a.g[g].first,
                       counts);
    MHIP_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_bj_fc, dim3(total([](const BjGroup& g) { return (g.npad / SB) * (g.npad / SB); })),
                     dim3(UPD_NT), 0, s, a, bst);
  MHIP_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_bj_ctf, dim3(total(tiles)), dim3(UPD_NT), 0, s, a, bst);
  MHIP_LAUNCH_CHECK();
  int open = 0;
  for (int sw = 0; sw <= max_sweeps; ++sw) {
    hipLaunchKernelGGL(k_bj_test, dim3(nmol), dim3(1024), 0, s, a, sw, sw == max_sweeps ? 1 : 0,
                       counts + 1 + sw);
    MHIP_LAUNCH_CHECK();
    MHIP_CHECK(hipMemcpyAsync(j->host, counts, sizeof(int) * (kMaxSweeps + 2), hipMemcpyDeviceToHost, s));
    MHIP_CHECK(hipEventRecord(j->tested, s));
    // the sweep's first launches find on the device which molecules go on, and
    // run while the host learns whether any does
    const BjLaunch whole = a;
    auto step = [&] {
      for (int g = 0; g < kGroups; ++g) a.on[g] = whole.on[g] && a.step < a.g[g].nsteps;
      const int wgs = total([](const BjGroup& g) { return g.npairs + g.ntiles + g.nctiles; });
      hipLaunchKernelGGL(k_bj_step, dim3(wgs), dim3(CROSS_THREADS), 0, s, a);
      MHIP_LAUNCH_CHECK();
    };
    a.step = 0;
    if (sw < max_sweeps) {
      if (sw == 0) {
        hipLaunchKernelGGL(k_bj_first, dim3(total([](const BjGroup& g) { return g.npairs; })), dim3(CROSS_THREADS), 0,
                           s, a);
        MHIP_LAUNCH_CHECK();
      }
      step();
    }
    MHIP_CHECK(hipEventSynchronize(j->tested));
    open = j->host[0];
    if (j->host[1 + sw] == 0) {
      a = whole;
      break;
    }
    for (; a.step < nsteps; ++a.step) {
      if (a.step > 0) step();
      for (int g = 0; g < kGroups; ++g)
        if (a.on[g]) a.par[g] ^= 1;
    }
    for (int g = 0; g < kGroups; ++g) a.on[g] = whole.on[g];
  }
  hipLaunchKernelGGL(k_bj_order, dim3(nmol), dim3(512), 0, s, a, bst);
  MHIP_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_bj_density, dim3(total(tiles)), dim3(UPD_NT), 0, s, a);
  MHIP_LAUNCH_CHECK();
  return open;
}

}  // namespace mhip
