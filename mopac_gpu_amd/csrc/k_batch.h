// A molecule of the batched SCF on the device, and the whole SCF of molecules
// in one workgroup each (k_batch.hip).
#pragma once
#include "common.h"
#include "k_fock.h"

namespace mhip {

struct BatchMol {
  int n, nocc, numat;
  double* f;
  double* p;
  double* pa;
  double* pold;
  double* p1;
  double* C;
  double* A;
  double* T;
  double* eig;
  double* fexit;  // packed scratch of the exit diagonalization (null: none)
};

struct BatchState {
  int niter, iredy, ready, done, converged, newdg, oknewd, recompute, have_c, do_eig, mode, itrmax;
  int adaptive;   // loosen the eigensolver's tolerance while PL is large
  int sweeps, ndiag, last_sweeps;  // Jacobi sweeps and diagonalizations so far
  int stuck;      // an eigensolve ran out of sweeps: the molecule does not count as converged
  int max_sweeps;
  double ten, shift, shfmax, shfto, shftbo, shiftb, pl, eold, diff, sellim, escf, ee;
  double eig_homo, eig_lumo, enuclr, atheat, selcon, pltest;
  // eigensolver work of this molecule since the batch was reset: applied
  // rotations, and FP64 flops of the method (12 n per rotation: 6 n on the
  // symmetric A, 6 n on C; warm start 2 n^3 + 2 n tri(n); density
  // 2 tri(n) nocc)
  long long eig_rot;
  double eig_flops;
};

// Up to this many orbitals; up to the second, one workgroup does the whole SCF.
constexpr int kMaxBatchN = 256;
constexpr int kMaxLdsN = 64;

constexpr int kEigSweeps = 60;  // the sweep limit of an eigensolve, at most

// The starting control state of one molecule (iter.F90:91-251).
BatchState batch_start(double enuclr, double atheat, double scfcrt, int itrmax);

// One molecule's SCF from P, Pa, pold and p1 in place, to self-consistency or
// itrmax, and its exit diagonalization to 1e-12 with phase_lock; mol and st are
// device pointers to one entry each.  Returns false, with nothing done, when
// the molecule does not fit the one-workgroup form.
bool scf_one_workgroup(hipStream_t s, int n, const FockArgs* args, const BatchMol* mol, BatchState* st, double tol,
                       int phase_lock);

// Block-Jacobi eigensolver of the molecules `which` of a batch (65 to 256
// orbitals), several workgroups to each (k_batch_eig.hip).
struct BatchJacobi;
BatchJacobi* bj_create(const std::vector<BatchMol>& mol, const std::vector<int>& which);
void bj_destroy(BatchJacobi* j);
// Diagonalizes the molecules with do_eig set whose padded size is in [lo, hi]:
// levels, eigenvectors (the next call's warm start) and the packed density.
// Waits for the device once a sweep; returns how many of them are not done.
int bj_solve(BatchJacobi* j, hipStream_t s, BatchState* bst, const int* do_eig, double tol, int max_sweeps, int lo,
             int hi);

}  // namespace mhip
