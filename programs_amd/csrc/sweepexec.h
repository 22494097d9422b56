// Device side of the one-launch triangular sweeps: the tables of a
// SweepPlan in HBM and the launches that use them (sweep.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "sweepplan.h"

namespace fvk {

// A launch runs unless every one of the n flags is set (stride in ints).
struct SweepGate {
  const int *done = nullptr;
  int stride = 0, n = 0;
};

struct SweepExec {
  int n = 0, P = 0, MW = 0, np = 0, slots = 0, width = kChunk, n_cu = 256, blocks = 0;  // blocks: launch size, 0: what fits
  size_t lds_[4] = {0, 0, 0, 0};
  bool bricks = false;
  std::vector<void *> mem;
  int *part = nullptr, *prow = nullptr, *ppos = nullptr;
  unsigned short *pslot = nullptr;
  struct Dir {
    int NE = 0;
    unsigned short *rec = nullptr;
    int *val = nullptr, *hsrc = nullptr;
    double *E = nullptr;       // exported values, 3 x NE; kSweepMark outside a sweep of this direction
    double *a = nullptr;       // MW x np entry values by position
  } d[2];
  int *tval = nullptr;
  double *aT = nullptr;        // MW x np transposed lower entries
  double *c = nullptr;         // factor by position (np)
  double *cr = nullptr;        // the backward sweep's row scale, rows in part order (n)
  double *Ec = nullptr;        // exported values of the factorisation (NE of d[0])
  double *t = nullptr;         // forward sweep's result, rows in part order (3 x n)
  int *ticket = nullptr;       // forward, backward, factor
  bool built = false;          // all of the above is there
  bool deny = false;           // the next build finds no memory (a test of that)
};

// Not built when there is no device memory for the tables (the caller then
// takes another form) or on an error; nothing is left allocated then.
int sweep_exec_build(SweepExec &X, const SweepPlan &p, hipStream_t s);
void sweep_exec_free(SweepExec &X);

// The matrix by position: entry values vals[val index], transposed lower
// entries tvals[...] (may be null: not needed by factor kind 0).  Opens the
// export buffer of a factorisation.
int sweep_pack(SweepExec &X, hipStream_t s, const double *vals, const double *tvals);
// The lower entries alone: vals[val index], or by the transposed entries'
// indices vals[tval]
int sweep_lower(SweepExec &X, hipStream_t s, const double *vals, bool transposed);
enum { SWEEP_DIC = 0, SWEEP_DILU = 1, SWEEP_FL = 2 };
// The factor of the packed matrix (sweep_pack before each): c = 1/(d+small)
// by row to crow, d to drow (null: not wanted); diag[dix ? dix[row] : row].
int sweep_factor(SweepExec &X, hipStream_t s, int kind, const double *diag, const int *dix, double *crow, double *drow,
                 int *err);
// The factor from row-ordered c and d (as solv_precond returns them)
int sweep_factor_from(SweepExec &X, hipStream_t s, const double *crow, const double *drow);
// x = M^-1 b for nc right-hand sides (component stride n), both sweeps
int sweep_apply(SweepExec &X, hipStream_t s, int nc, const double *b, double *x, SweepGate gate, int *err);

}  // namespace fvk
