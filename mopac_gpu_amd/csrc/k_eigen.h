// Block-Jacobi symmetric eigensolver (k_eigen.hip).
#pragma once
#include "common.h"

namespace mhip {

struct JacobiPlan {
  int n = 0, npad = 0, nb = 0, npairs = 0;
  int nsteps = 0;        // steps per sweep
  bool grouped = false;  // pairs only within [0, split) and [split, n)
  int split = 0;
  int npo = 0;  // pairs of the first group in every step (npairs when not grouped)
  int max_inner = 0;  // inner Jacobi sweeps per 64x64 pair problem (0: by the schedule)
  // Optional HIP-event timing of the solve and A-update launches.
  bool timing = false;
  double t_solve_ms = 0.0, t_apply_ms = 0.0, t_applyc_ms = 0.0;
  long long n_solve = 0, n_apply = 0, n_applyc = 0;
  long long active_tiles = 0, active_pairs = 0;  // summed over timed launches
  long long active_rotations = 0;                 // 2x2 rotations of the timed solves
  std::vector<int> intra_host;                    // host copy of intra
  std::vector<hipEvent_t> ev;
  hipEvent_t tested = nullptr;                    // behind the last stopping test
  void ensure_test_event(hipStream_t s);
  DevBuf pairs;  // nsteps x npairs x 2 block indices
  DevBuf qbuf;   // two steps x npairs x 64 x 64 rotations
  DevBuf diag;   // two steps x nb x 32 x 32 diagonal blocks as the solves left them
  DevBuf where;  // nsteps x nb: 2 x (pair of the block in the step) + half
  DevBuf part;   // reduction scratch
  DevBuf perm;   // sort permutation
  DevBuf active; // two steps x npairs: 1 when Q != I
  DevBuf intra;  // nsteps x npairs: 1 where the cross-round solve also
                 // rotates inside the two blocks (once per sweep of a group)
  DevBuf counts; // active pairs per step (timing mode)
  // split > 0 (a multiple of 32 leaving an even number of blocks on both
  // sides): rotations only within the leading split columns and within the
  // rest, for a matrix already block-diagonal in that partition.
  void build(int n, int split = 0);
  void release() {
    for (DevBuf* b : {&pairs, &qbuf, &diag, &where, &part, &perm, &active, &intra, &counts}) b->release();
    for (auto e : ev) (void)hipEventDestroy(e);
    ev.clear();
    if (tested) (void)hipEventDestroy(tested);
    tested = nullptr;
  }
};

// Pair-solve schedule of every plan in the process: 1 (default) = cross
// rounds with one intra-block pass per sweep, 0 = a full 64-index cyclic
// sweep in every step.
extern int g_jacobi_schedule;

void jacobi_set_identity(hipStream_t s, int npad, double* C, int ldc);
// Sweeps until max|offdiag| <= tol * max(1, max|diag|).  A2 is scratch of A's
// size; the steps go from one to the other, and A names the one that holds
// the result on return.  With c_blocks (a grouped plan) C is two diagonal
// blocks, the rest of it zero and left alone.  host_scal: two doubles in
// pinned memory.  Returns 0 when converged, 1 when max_sweeps ran out.
int jacobi_sweeps(hipStream_t s, JacobiPlan& plan, double*& A, double*& A2, double* C, double tol, int max_sweeps,
                  double* host_scal, double* dev_scal, int* sweeps_done, bool c_blocks = false);
// eig_dev[k] = k-th smallest diagonal entry, Cout[:,k] = C[:,perm[k]].
void jacobi_sort(hipStream_t s, JacobiPlan& plan, const double* A, const double* C, double* Cout,
                 double* eig_dev);
void phase_lock(hipStream_t s, int n, double* C, int ldc);

}  // namespace mhip
