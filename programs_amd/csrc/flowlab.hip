// flowlab's serial CSR SIMPLE on gfx950: geometry (geometry_m.f90:97-330),
// least-squares gradients (ls_grad_matrix / ls_gradient, :592-730),
// momentum and pressure-correction assembly (transport_m.f90:58-348,
// :430-629, ns_source :726-752, ns_correction :757-800) and the CSR Krylov
// solvers with their factor (solv_m.f90:10-289), on one device context
// built from the arrays flowlab's Fortran receives (flmesh.h).
//
// Data layout: cells in the reference's order (domain-local index), faces
// in the reference's face order, structure-of-arrays.  A sum the reference
// builds by scattering over faces in face order is gathered per cell over
// the cell's faces in ascending face order: the same additions in the same
// order, so the geometry, the gradients and the assembled matrices and
// right-hand sides equal the reference's bit for bit (compiled without FMA
// contraction).  The Krylov reductions run in a fixed tree (rounding-level
// differences from the reference's sequential sums).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "ctx.h"
#include "flmesh.h"
#include "sweep.h"

namespace fvk {

// ---------------------------------------------------------------- context
struct FlKS {  // scalars of one component's Krylov solve (solv_m.f90 cof(1:6))
  double cof[7];
  double norm, norm0;
  int iter, done, pad[2];
};

struct FlCtx {
  int device = 0;
  hipStream_t stream = nullptr;
  int nd = 0, n = 0, nb = 0, nf = 0, nnz = 0, n_vrt = 0;
  std::vector<void *> owned;
  HostIo io;
  std::vector<int> h_ia, h_ja, h_j1, h_jn, h_btag;
  // geometry
  double *xvc = nullptr, *vol = nullptr, *volr = nullptr, *ls = nullptr;
  double *xfc = nullptr, *nrm = nullptr, *area = nullptr, *xpc = nullptr, *xnc = nullptr, *lpn = nullptr,
         *wfp = nullptr, *fvol = nullptr;
  int *j1 = nullptr, *jn = nullptr, *btag = nullptr;
  // matrix pattern
  int *ia = nullptr, *ja = nullptr, *kii = nullptr, *kij = nullptr, *kji = nullptr, *tpos = nullptr;
  // a row's lower entries are [ia, klo) (the reference's loops stop at the
  // first column >= the row), its upper entries [kup, ia+1) (taken from the
  // end down to the first column <= the row)
  int *klo = nullptr, *kup = nullptr;
  int *cptr = nullptr, *cfl = nullptr;
  // triangular sweeps by levels (lower / upper dependencies)
  std::vector<int> lf_ptr, lb_ptr;
  int *lf_rows = nullptr, *lb_rows = nullptr;
  // one launch per factorisation / sweep (rows wait for their values) when
  // no row has more than kSweepSlots lower or upper entries
  bool one_launch = true;
  int n_cu = 256;
  int sweep_blocks = 0;  // blocks of the one-launch kernels (0: one per CU)
  // the default form: parts of rows, each walked by one block (sweep.hip)
  SweepExec sw;
  int parts = 0;         // 1: where they are the faster form, 2: always, 0: never
  int part_rows = 4096;  // rows of a part at most
  long positions = 0;    // positions of its tables at most (0: the kernels' limit)
  bool narrow = false;   // no row has more than kSweepSlots lower or upper entries
  std::vector<int> h_kii, h_klo, h_kup, h_tpos;
  int *sweep_int = nullptr;  // tickets: forward, backward, factor; [3] wait-bound error
  // Krylov work: 6 vectors x 3 components, partials, scalars
  double *wk = nullptr, *pc = nullptr, *part = nullptr;
  FlKS *ks = nullptr;
  // the matrix of a solve by slots (slot k of row i at k*n + i, column -1:
  // none) when no row has more than 8 entries; ew: slots, 0: CSR only
  int ew = 0;
  int *ecol = nullptr;
  double *eval = nullptr;
  DoneWatch watch;
  double *scal = nullptr;  // c_rat and scratch scalars
  // workspaces of the calls on host arrays, kept once made: matrix values,
  // solution and right-hand side; boundary values and boundary faces
  double *lin = nullptr, *bval = nullptr;
  int *bfl = nullptr;
  int n_bf = 0;
};

// zeroed allocation; the clear has finished when this returns (an upload
// that follows on another stream must not race it)
template <class T>
static int fl_alloc(FlCtx &c, T **p, size_t n) {
  void *q = nullptr;
  FVK_HIP(hipMalloc(&q, (n ? n : 1) * sizeof(T)));
  c.owned.push_back(q);
  FVK_HIP(hipMemsetAsync(q, 0, (n ? n : 1) * sizeof(T), c.stream));
  FVK_HIP(hipStreamSynchronize(c.stream));
  *p = (T *)q;
  return 0;
}
template <class T>
static int fl_up(FlCtx &c, T **p, const std::vector<T> &v) {
  int rc = fl_alloc(c, p, v.size());
  if (rc) return rc;
  if (!v.empty()) FVK_HIP(hipMemcpy(*p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  return 0;
}

static void fl_free(FlCtx &c, void *p) {
  if (!p) return;
  for (size_t k = 0; k < c.owned.size(); ++k)
    if (c.owned[k] == p) {
      hipFree(p);
      c.owned.erase(c.owned.begin() + (long)k);
      return;
    }
}

static double *wkv(FlCtx &c, int k) { return c.wk + (size_t)k * 3 * c.n; }

// ---------------------------------------------------------------- geometry
// cross_prod (vector_utils_m.f90:35-41)
__device__ __forceinline__ void fl_cross(const double *a, const double *b, double *v) {
  v[0] = a[1] * b[2] - b[1] * a[2];
  v[1] = a[2] * b[0] - b[2] * a[0];
  v[2] = a[0] * b[1] - b[0] * a[1];
}

__global__ __launch_bounds__(BS) void k_fl_centre(int n, int nd, const double *__restrict__ xv,
                                                  const int *__restrict__ evp, const int *__restrict__ evr,
                                                  double *__restrict__ xvc) {
  const int i = blockIdx.x * BS + threadIdx.x;
  if (i >= n) return;
  double x[3] = {0.0, 0.0, 0.0};
  const int a = evp[i], b = evp[i + 1];
  for (int k = a; k < b; ++k)
    for (int d = 0; d < nd; ++d) x[d] = x[d] + xv[3 * (size_t)evr[k] + d];
  const double cnt = (double)(b - a);
  for (int d = 0; d < nd; ++d) xvc[(size_t)d * n + i] = x[d] / cnt;
}

// geometry_m.f90:140-300 for one face
__global__ __launch_bounds__(BS) void k_fl_face_geom(int nf, int n, int nd, const double *__restrict__ xv,
                                                     const int *__restrict__ fvp, const int *__restrict__ fvr,
                                                     const int *__restrict__ j1, const int *__restrict__ jn,
                                                     const double *__restrict__ xvc, double *xfc, double *nrm,
                                                     double *area, double *xpc, double *xnc, double *lpn,
                                                     double *wfp, double *fvol) {
  const int f = blockIdx.x * BS + threadIdx.x;
  if (f >= nf) return;
  const int a = fvp[f], b = fvp[f + 1], nv = b - a;
  double x1[3] = {0.0, 0.0, 0.0};
  for (int k = a; k < b; ++k)
    for (int d = 0; d < nd; ++d) x1[d] = x1[d] + xv[3 * (size_t)fvr[k] + d];
  double xf[3] = {0.0, 0.0, 0.0};
  for (int d = 0; d < nd; ++d) xf[d] = x1[d] / (double)nv;
  // face normal and area
  const double *v0 = xv + 3 * (size_t)fvr[a];
  double s[3] = {0.0, 0.0, 0.0}, e1[3] = {0.0, 0.0, 0.0};
  for (int k = a + 1; k < b; ++k) {
    double e[3] = {0.0, 0.0, 0.0};
    const double *vk = xv + 3 * (size_t)fvr[k];
    for (int d = 0; d < nd; ++d) e[d] = vk[d] - v0[d];
    if (nv == 2) {
      const double uz[3] = {0.0, 0.0, 1.0};
      double cp[3];
      fl_cross(e, uz, cp);
      for (int d = 0; d < nd; ++d) s[d] = cp[d];
    } else {
      if (k - (a + 1) >= 1) {
        double cp[3];
        fl_cross(e1, e, cp);
        for (int d = 0; d < 3; ++d) s[d] = s[d] + 0.5 * cp[d];
      }
      for (int d = 0; d < 3; ++d) e1[d] = e[d];
    }
  }
  double ss = 0.0;
  for (int d = 0; d < nd; ++d) ss = ss + s[d] * s[d];
  const double ar = sqrt(ss);
  double nv3[3] = {0.0, 0.0, 0.0};
  for (int d = 0; d < nd; ++d) nv3[d] = s[d] / ar;
  area[f] = ar;
  for (int d = 0; d < nd; ++d) {
    xfc[(size_t)d * nf + f] = xf[d];
    nrm[(size_t)d * nf + f] = nv3[d];
  }
  fvol[f] = xf[0] * nv3[0] * ar;
  const int p = j1[f];
  double dx[3], t = 0.0;
  for (int d = 0; d < nd; ++d) dx[d] = xf[d] - xvc[(size_t)d * n + p];
  for (int d = 0; d < nd; ++d) t = t + dx[d] * nv3[d];
  double xp[3];
  for (int d = 0; d < nd; ++d) {
    xp[d] = xf[d] - nv3[d] * t;
    xpc[(size_t)d * nf + f] = xp[d];
  }
  const int q = jn[f];
  if (q >= 0) {
    double u = 0.0, xn[3];
    for (int d = 0; d < nd; ++d) dx[d] = xf[d] - xvc[(size_t)d * n + q];
    for (int d = 0; d < nd; ++d) u = u + dx[d] * nv3[d];
    for (int d = 0; d < nd; ++d) {
      xn[d] = xf[d] - nv3[d] * u;
      xnc[(size_t)d * nf + f] = xn[d];
    }
    double l = 0.0, w = 0.0;
    for (int d = 0; d < nd; ++d) l = l + (xn[d] - xp[d]) * (xn[d] - xp[d]);
    const double l_pn = sqrt(l);
    for (int d = 0; d < nd; ++d) w = w + (xf[d] - xp[d]) * (xf[d] - xp[d]);
    wfp[f] = sqrt(w) / l_pn;
    lpn[f] = l_pn;
  } else {
    double l = 0.0;
    for (int d = 0; d < nd; ++d) l = l + (xf[d] - xp[d]) * (xf[d] - xp[d]);
    lpn[f] = sqrt(l);
  }
}

// volume: the face scatter of geometry_m.f90:212-232 gathered per cell
__global__ __launch_bounds__(BS) void k_fl_vol(int n, const int *__restrict__ cptr, const int *__restrict__ cfl,
                                               const int *__restrict__ j1, const double *__restrict__ fvol,
                                               double *vol, double *volr) {
  const int i = xcd_block() * BS + threadIdx.x;
  if (i >= n) return;
  double v = 0.0;
  for (int k = cptr[i]; k < cptr[i + 1]; ++k) {
    const int f = cfl[k];
    v = j1[f] == i ? v + fvol[f] : v - fvol[f];
  }
  vol[i] = v;
  volr[i] = 1.0 / (v + SMALL);
}

// matrix_inv (matrix_utils_m.f90:8-52) of a column-major nd x nd matrix
__device__ __forceinline__ void fl_inv(int nd, const double *m, double *inv) {
#define M(i, j) m[((j) - 1) * nd + (i) - 1]
#define I(i, j) inv[((j) - 1) * nd + (i) - 1]
  double det;
  if (nd == 2) {
    det = M(1, 1) * M(2, 2) - M(1, 2) * M(2, 1);
  } else {
    det = (M(2, 2) * M(3, 3) - M(2, 3) * M(3, 2)) * M(1, 1);
    det = det + (M(2, 3) * M(3, 1) - M(2, 1) * M(3, 3)) * M(1, 2);
    det = det + (M(2, 1) * M(3, 2) - M(2, 2) * M(3, 1)) * M(1, 3);
  }
  if (fabs(det) < SMALL) {
    for (int k = 0; k < nd * nd; ++k) inv[k] = 0.0;
    return;
  }
  if (nd == 2) {
    I(1, 1) = M(2, 2);
    I(1, 2) = -M(1, 2);
    I(2, 1) = -M(2, 1);
    I(2, 2) = M(1, 1);
  } else {
    I(1, 1) = M(2, 2) * M(3, 3) - M(2, 3) * M(3, 2);
    I(2, 1) = M(2, 3) * M(3, 1) - M(2, 1) * M(3, 3);
    I(3, 1) = M(2, 1) * M(3, 2) - M(2, 2) * M(3, 1);
    I(1, 2) = M(3, 2) * M(1, 3) - M(3, 3) * M(1, 2);
    I(2, 2) = M(3, 3) * M(1, 1) - M(3, 1) * M(1, 3);
    I(3, 2) = M(3, 1) * M(1, 2) - M(3, 2) * M(1, 1);
    I(1, 3) = M(1, 2) * M(2, 3) - M(1, 3) * M(2, 2);
    I(2, 3) = M(1, 3) * M(2, 1) - M(1, 1) * M(2, 3);
    I(3, 3) = M(1, 1) * M(2, 2) - M(1, 2) * M(2, 1);
  }
  for (int k = 0; k < nd * nd; ++k) inv[k] = inv[k] / det;
#undef M
#undef I
}

// ls_grad_matrix (geometry_m.f90:592-660): sum of dx dx^T over the cell's
// faces (ascending), inverted; ls[(jc*nd + ic)*n + i] = inverse(ic, jc)
__global__ __launch_bounds__(BS) void k_fl_ls(int n, int nf, int nd, const int *__restrict__ cptr,
                                              const int *__restrict__ cfl, const int *__restrict__ j1,
                                              const int *__restrict__ jn, const double *__restrict__ xvc,
                                              const double *__restrict__ xfc, double *ls) {
  const int i = xcd_block() * BS + threadIdx.x;
  if (i >= n) return;
  double m[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int k = cptr[i]; k < cptr[i + 1]; ++k) {
    const int f = cfl[k], p = j1[f], q = jn[f];
    double dx[3];
    for (int d = 0; d < nd; ++d)
      dx[d] = q >= 0 ? xvc[(size_t)d * n + q] - xvc[(size_t)d * n + p] : xfc[(size_t)d * nf + f] - xvc[(size_t)d * n + p];
    for (int jc = 0; jc < nd; ++jc)
      for (int ic = 0; ic < nd; ++ic) m[jc * nd + ic] = m[jc * nd + ic] + dx[ic] * dx[jc];
  }
  double inv[9];
  fl_inv(nd, m, inv);
  for (int k = 0; k < nd * nd; ++k) ls[(size_t)k * n + i] = inv[k];
}

// ---------------------------------------------------------------- gradients
// ls_gradient (geometry_m.f90:665-770): g(:, q) = LS * sum over faces of
// dx dphi(q); neu: boundary differences are zero and the boundary values
// are extrapolated afterwards (k_fl_grad_bnd)
__global__ __launch_bounds__(BS) void k_fl_grad(int n, int nf, int nb, int nd, int ncmp, const int *__restrict__ cptr,
                                                const int *__restrict__ cfl, const int *__restrict__ j1,
                                                const int *__restrict__ jn, const double *__restrict__ xvc,
                                                const double *__restrict__ xfc, const double *__restrict__ ls,
                                                const double *__restrict__ phi, const double *__restrict__ phib,
                                                int neu, double *__restrict__ g) {
  const int i = xcd_block() * BS + threadIdx.x;
  if (i >= n) return;
  double a[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};  // a[q][d]
  for (int k = cptr[i]; k < cptr[i + 1]; ++k) {
    const int f = cfl[k], p = j1[f], q = jn[f];
    double dx[3], dp[3];
    if (q >= 0) {
      for (int d = 0; d < nd; ++d) dx[d] = xvc[(size_t)d * n + q] - xvc[(size_t)d * n + p];
      for (int c = 0; c < ncmp; ++c) dp[c] = phi[(size_t)c * n + q] - phi[(size_t)c * n + p];
    } else {
      const int b = -q - 1;
      for (int d = 0; d < nd; ++d) dx[d] = xfc[(size_t)d * nf + f] - xvc[(size_t)d * n + p];
      for (int c = 0; c < ncmp; ++c) dp[c] = neu ? 0.0 : phib[(size_t)c * nb + b] - phi[(size_t)c * n + p];
    }
    for (int c = 0; c < ncmp; ++c)
      for (int d = 0; d < nd; ++d) a[c][d] = a[c][d] + dx[d] * dp[c];
  }
  double L[9];
  for (int k = 0; k < nd * nd; ++k) L[k] = ls[(size_t)k * n + i];
  for (int c = 0; c < ncmp; ++c)
    for (int r = 0; r < nd; ++r) {
      double s = 0.0;
      for (int j = 0; j < nd; ++j) s = s + L[j * nd + r] * a[c][j];
      g[(size_t)(c * nd + r) * n + i] = s;
    }
}

__global__ __launch_bounds__(BS) void k_fl_grad_bnd(int nbf, const int *__restrict__ bfl, int n, int nf, int nb,
                                                    int nd, int ncmp, const int *__restrict__ j1,
                                                    const int *__restrict__ jn, const double *__restrict__ xvc,
                                                    const double *__restrict__ xfc, const double *__restrict__ phi,
                                                    const double *__restrict__ g, double *phib) {
  const int t = blockIdx.x * BS + threadIdx.x;
  if (t >= nbf) return;
  const int f = bfl[t], p = j1[f], b = -jn[f] - 1;
  double dx[3];
  for (int d = 0; d < nd; ++d) dx[d] = xfc[(size_t)d * nf + f] - xvc[(size_t)d * n + p];
  for (int c = 0; c < ncmp; ++c) {
    double s = 0.0;
    for (int d = 0; d < nd; ++d) s = s + g[(size_t)(c * nd + d) * n + p] * dx[d];
    phib[(size_t)c * nb + b] = phi[(size_t)c * n + p] + s;
  }
}

// ---------------------------------------------------------------- Krylov
// The matrix of a solve.  A thread per row of the CSR arrays reads addresses
// a row apart; by slots neighbouring threads read neighbouring addresses.
struct FlMat {
  int n;
  const int *ia, *ja, *ecol;
  const double *a, *eval;
};

__global__ __launch_bounds__(BS) void k_fl_slots(FlMat M, int ew, int *__restrict__ ecol, double *__restrict__ eval) {
  const int i = blockIdx.x * BS + threadIdx.x;
  if (i >= M.n) return;
  const int k0 = M.ia[i], nk = M.ia[i + 1] - k0;
  for (int k = 0; k < ew; ++k) {
    const size_t o = (size_t)k * M.n + i;
    if (ecol) ecol[o] = k < nk ? M.ja[k0 + k] : -1;
    if (eval) eval[o] = k < nk ? M.a[k0 + k] : 0.0;
  }
}

// csr_matvec_prod (matrix_utils_m.f90:70-82): y(i) = 0 + sum a x in CSR
// order, x(q, j) the value of component q at row j; WS: slots, 0: CSR
template <int NC, int WS, class X>
__device__ __forceinline__ void fl_row_mv(const FlMat &M, int i, X x, double (&y)[NC]) {
#pragma unroll
  for (int q = 0; q < NC; ++q) y[q] = 0.0;
  if (WS > 0) {
#pragma unroll
    for (int k = 0; k < WS; ++k) {
      const size_t o = (size_t)k * M.n + i;
      const int j = M.ecol[o];
      const double a = M.eval[o];
      if (j >= 0)
#pragma unroll
        for (int q = 0; q < NC; ++q) y[q] = y[q] + a * x(q, j);
    }
  } else {
    for (int k = M.ia[i]; k < M.ia[i + 1]; ++k) {
      const int j = M.ja[k];
      const double a = M.a[k];
#pragma unroll
      for (int q = 0; q < NC; ++q) y[q] = y[q] + a * x(q, j);
    }
  }
}

// preconditioner (solv_m.f90:224-250) over one level of rows
__global__ __launch_bounds__(BS) void k_fl_pc_level(const int *__restrict__ rows, int cnt, const int *__restrict__ ia,
                                                    const int *__restrict__ ja, const int *__restrict__ kii,
                                                    const int *__restrict__ tpos, const double *__restrict__ a,
                                                    double *pc) {
  const int t = blockIdx.x * BS + threadIdx.x;
  if (t >= cnt) return;
  const int i = rows[t];
  double s = a[kii[i]];
  for (int k = ia[i]; k < ia[i + 1]; ++k) {
    const int j = ja[k];
    if (j >= i) break;
    s = s - a[k] * pc[j] * a[tpos[k]];
  }
  pc[i] = 1.0 / (s + SMALL);
}

// direct_solve forward sweep (solv_m.f90:255-268) for ncmp right-hand sides
__global__ __launch_bounds__(BS) void k_fl_fwd_level(const int *__restrict__ rows, int cnt, int n, int ncmp,
                                                     const int *__restrict__ ia, const int *__restrict__ ja,
                                                     const double *__restrict__ a, const double *__restrict__ pc,
                                                     const double *__restrict__ b, double *x,
                                                     const FlKS *__restrict__ ks) {
  const int t = blockIdx.x * BS + threadIdx.x;
  if (t >= cnt) return;
  const int i = rows[t];
  for (int c = 0; c < ncmp; ++c) {
    if (ks && ks[c].done) continue;
    double s = b[(size_t)c * n + i];
    for (int k = ia[i]; k < ia[i + 1]; ++k) {
      const int j = ja[k];
      if (j >= i) break;
      s = s - a[k] * x[(size_t)c * n + j];
    }
    x[(size_t)c * n + i] = s * pc[i];
  }
}

// direct_solve scaling and backward sweep (solv_m.f90:270-286): t holds the
// forward result, y receives x
__global__ __launch_bounds__(BS) void k_fl_bwd_level(const int *__restrict__ rows, int cnt, int n, int ncmp,
                                                     const int *__restrict__ ia, const int *__restrict__ ja,
                                                     const double *__restrict__ a, const double *__restrict__ pc,
                                                     const double *__restrict__ tf, double *y,
                                                     const FlKS *__restrict__ ks) {
  const int t = blockIdx.x * BS + threadIdx.x;
  if (t >= cnt) return;
  const int i = rows[t];
  const double cof = 1.0 / (pc[i] + SMALL);
  for (int c = 0; c < ncmp; ++c) {
    if (ks && ks[c].done) continue;
    double s = cof * tf[(size_t)c * n + i];
    for (int k = ia[i + 1] - 1; k >= ia[i]; --k) {
      const int j = ja[k];
      if (j <= i) break;
      s = s - a[k] * y[(size_t)c * n + j];
    }
    y[(size_t)c * n + i] = s * pc[i];
  }
}

// The Krylov kernels leave a partial per block of NC (or NC pairs of) sums;
// the kernel that uses a sum adds the partials itself, every block in the same
// tree, so that a scalar step costs no launch of its own.  Only the end of an
// iteration is a launch (k_fl_end): the sweeps after it are skipped once every
// component is done.  A CG iteration takes 6 launches, a BiCGStab iteration
// 10; with a launch per scalar step they were 9 and 15, and on the momentum
// systems, which end after one iteration, most of them found nothing to do
// (96^3, three outer iterations: 38.3 -> 30.4 ms; there the products by slots
// take 24.9 us with the direction update, by CSR they took 35.6 us without).
__device__ __forceinline__ bool fl_all_done(const FlKS *ks, int ncmp) {
  if (!ks) return false;
  for (int c = 0; c < ncmp; ++c)
    if (!ks[c].done) return false;
  return true;
}

// f(component, index into a vector's components, row) for this block's rows
// of the components that are not done
template <int NC, class F>
__device__ __forceinline__ void fl_rows(int n, const int (&dn)[NC], F f) {
  int r0, r1;
  block_rows<RB>(n, r0, r1);
  for (int i = r0 + (int)threadIdx.x; i < r1; i += RB)
#pragma unroll
    for (int q = 0; q < NC; ++q)
      if (!dn[q]) f(q, (size_t)q * n + i);
}
template <int NC>
__device__ __forceinline__ bool fl_open(const FlKS *ks, int (&dn)[NC]) {
  bool any = false;
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    dn[q] = ks[q].done;
    any = any || !dn[q];
  }
  return any;
}

// initial residual: res = res - A phi; w1 = res; sums |res| and (BiCGStab)
// res.res; the search direction p (and u) start at zero
template <int NC, int WS>
__global__ __launch_bounds__(RB) void k_fl_init(FlMat M, const double *__restrict__ phi, double *res, double *w1,
                                                double *p, double *u, double *part) {
  const int n = M.n;
  double v[2 * NC];
#pragma unroll
  for (int q = 0; q < 2 * NC; ++q) v[q] = 0.0;
  int r0, r1;
  block_rows<RB>(n, r0, r1);
  for (int i = r0 + (int)threadIdx.x; i < r1; i += RB) {
    double y[NC];
    fl_row_mv<NC, WS>(M, i, [&](int q, int j) { return phi[(size_t)q * n + j]; }, y);
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      const size_t o = (size_t)q * n + i;
      const double r = res[o] - y[q];
      res[o] = r;
      w1[o] = r;
      p[o] = 0.0;
      if (u) u[o] = 0.0;
      v[q] += fabs(r);
      v[NC + q] += r * r;
    }
  }
  store_partials<2 * NC, RB>(v, part);
}

// sum x.y
template <int NC>
__global__ __launch_bounds__(RB) void k_fl_dot(int n, const double *__restrict__ x, const double *__restrict__ y,
                                               const FlKS *ks, double *part) {
  int dn[NC];
  if (!fl_open<NC>(ks, dn)) return;
  double v[NC];
#pragma unroll
  for (int q = 0; q < NC; ++q) v[q] = 0.0;
  fl_rows<NC>(n, dn, [&](int q, size_t o) { v[q] += x[o] * y[o]; });
  store_partials<NC, RB>(v, part);
}

// CG: beta from z.r (partS) ; p = z + beta p ; q = A p ; sum p.q.  The
// neighbours' p is formed from z and the old p.  cof[0]: z.r for k_fl_end
// (the other blocks still read the old one, cof[4]).
template <int NC, int WS>
__global__ __launch_bounds__(RB) void k_fl_cg_pq(FlMat M, const double *__restrict__ z, const double *__restrict__ pold,
                                                 double *__restrict__ pnew, double *__restrict__ qv,
                                                 const double *__restrict__ partS, int P, FlKS *ks, double *part) {
  int dn[NC];
  if (!fl_open<NC>(ks, dn)) return;
  const int n = M.n;
  double s[NC], beta[NC], v[NC];
  load_totals<NC, RB>(partS, P, s);
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    beta[q] = 1.0 / (ks[q].cof[4] + SMALL);
    beta[q] = beta[q] * s[q];
    v[q] = 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0 && !dn[q]) ks[q].cof[0] = s[q];
  }
  int r0, r1;
  block_rows<RB>(n, r0, r1);
  for (int i = r0 + (int)threadIdx.x; i < r1; i += RB) {
    double y[NC];
    fl_row_mv<NC, WS>(M, i, [&](int q, int j) {
      const size_t o = (size_t)q * n + j;
      return z[o] + beta[q] * pold[o];
    }, y);
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      if (dn[q]) continue;
      const size_t o = (size_t)q * n + i;
      const double pi = z[o] + beta[q] * pold[o];
      pnew[o] = pi;
      qv[o] = y[q];
      v[q] += pi * y[q];
    }
  }
  store_partials<NC, RB>(v, part);
}

// CG: alpha = z.r / p.q (partQ) ; phi += alpha p ; r -= alpha q ; sum |r|
template <int NC>
__global__ __launch_bounds__(RB) void k_fl_cg_upd(int n, double *__restrict__ phi, const double *__restrict__ p,
                                                  double *__restrict__ r, const double *__restrict__ qv,
                                                  const double *__restrict__ partQ, int P, const FlKS *ks,
                                                  double *part) {
  int dn[NC];
  if (!fl_open<NC>(ks, dn)) return;
  double t[NC], al[NC], v[NC];
  load_totals<NC, RB>(partQ, P, t);
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    al[q] = ks[q].cof[0] / (t[q] + SMALL);
    v[q] = 0.0;
  }
  fl_rows<NC>(n, dn, [&](int q, size_t o) {
    phi[o] = phi[o] + al[q] * p[o];
    const double rr = r[o] - al[q] * qv[o];
    r[o] = rr;
    v[q] += fabs(rr);
  });
  store_partials<NC, RB>(v, part);
}

// BiCGStab: p = r + omega (p - alpha u)
template <int NC>
__global__ __launch_bounds__(BS) void k_fl_bi_dir(int n, double *p, const double *__restrict__ r,
                                                  const double *__restrict__ u, const FlKS *ks) {
  const int i = blockIdx.x * BS + threadIdx.x;
  if (i >= n) return;
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    if (ks[q].done) continue;
    const size_t o = (size_t)q * n + i;
    p[o] = r[o] + ks[q].cof[6] * (p[o] - ks[q].cof[2] * u[o]);
  }
}

// BiCGStab: y = A z ; sum y.d, and with SQ sum (y + small)^2 (solv_m.f90:190-196)
template <int NC, int WS, bool SQ>
__global__ __launch_bounds__(RB) void k_fl_bi_mv(FlMat M, const double *__restrict__ z, double *__restrict__ y,
                                                 const double *__restrict__ d, const FlKS *ks, double *part) {
  int dn[NC];
  if (!fl_open<NC>(ks, dn)) return;
  const int n = M.n;
  constexpr int NV = SQ ? 2 * NC : NC;
  double v[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) v[q] = 0.0;
  int r0, r1;
  block_rows<RB>(n, r0, r1);
  for (int i = r0 + (int)threadIdx.x; i < r1; i += RB) {
    double w[NC];
    fl_row_mv<NC, WS>(M, i, [&](int q, int j) { return z[(size_t)q * n + j]; }, w);
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      if (dn[q]) continue;
      const size_t o = (size_t)q * n + i;
      y[o] = w[q];
      v[q] += w[q] * d[o];
      if (SQ) v[NV - NC + q] += (w[q] + SMALL) * (w[q] + SMALL);
    }
  }
  store_partials<NV, RB>(v, part);
}

// BiCGStab, first half: gamma = beta / u.r0 (partT) ; phi += gamma z ;
// r -= gamma u
template <int NC>
__global__ __launch_bounds__(RB) void k_fl_bi_upd1(int n, double *__restrict__ phi, const double *__restrict__ z,
                                                   double *__restrict__ r, const double *__restrict__ u,
                                                   const double *__restrict__ partT, int P, FlKS *ks) {
  int dn[NC];
  if (!fl_open<NC>(ks, dn)) return;
  double t[NC], g[NC];
  load_totals<NC, RB>(partT, P, t);
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    g[q] = ks[q].cof[4] / (t[q] + SMALL);
    if (blockIdx.x == 0 && threadIdx.x == 0 && !dn[q]) ks[q].cof[5] = g[q];
  }
  fl_rows<NC>(n, dn, [&](int q, size_t o) {
    phi[o] = phi[o] + g[q] * z[o];
    r[o] = r[o] - g[q] * u[o];
  });
}

// BiCGStab, second half: alpha from partD ; phi += alpha z ; r -= alpha v ;
// sums |r| and r.r0 (the next iteration's beta)
template <int NC>
__global__ __launch_bounds__(RB) void k_fl_bi_upd2(int n, double *__restrict__ phi, const double *__restrict__ z,
                                                   double *__restrict__ r, const double *__restrict__ vv,
                                                   const double *__restrict__ r0v, const double *__restrict__ partD,
                                                   int P, FlKS *ks, double *part) {
  int dn[NC];
  if (!fl_open<NC>(ks, dn)) return;
  double t[2 * NC], al[NC], v[2 * NC];
  load_totals<2 * NC, RB>(partD, P, t);
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    al[q] = t[q] / (t[NC + q] + SMALL);
    v[q] = v[NC + q] = 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0 && !dn[q]) ks[q].cof[2] = al[q];
  }
  fl_rows<NC>(n, dn, [&](int q, size_t o) {
    phi[o] = phi[o] + al[q] * z[o];
    const double rr = r[o] - al[q] * vv[o];
    r[o] = rr;
    v[q] += fabs(rr);
    v[NC + q] += rr * r0v[o];
  });
  store_partials<2 * NC, RB>(v, part);
}

// The scalar steps between two iterations of cg_solver / bicg_solver (one
// block): the start (first) or the norm and the exit test, then for BiCGStab
// the next beta and omega.  part: NV totals per component, |r| and (BiCGStab,
// start) a second one.
template <int NC, bool BICG>
__global__ __launch_bounds__(RB) void k_fl_end(int first, int P, const double *__restrict__ part, FlKS *ks, double reduc,
                                               DoneSlot slot) {
  double t[2 * NC];
#pragma unroll
  for (int q = 0; q < 2 * NC; ++q) t[q] = 0.0;
  bool open = true;
  if (!first) open = !fl_all_done(ks, NC);
  if (open) {
    if (BICG) {
      load_totals<2 * NC, RB>(part, P, t);
    } else {
      double t1[NC];
      load_totals<NC, RB>(part, P, t1);
#pragma unroll
      for (int q = 0; q < NC; ++q) t[q] = t1[q];
    }
  }
  if (threadIdx.x != 0) return;
  bool all = true;
  if (open)
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      FlKS &k = ks[q];
      if (first) {
        for (int j = 0; j < 7; ++j) k.cof[j] = 0.0;
        k.norm = k.norm0 = t[q];
        k.iter = 0;
        k.done = 0;
        if (BICG) k.cof[2] = k.cof[3] = k.cof[5] = 1.0;
        else k.cof[4] = 1.0 / SMALL;
      } else {
        if (k.done) continue;
        k.norm = t[q];
        k.cof[1] = t[q] / (k.norm0 + SMALL);
        k.iter += 1;
        if (k.cof[1] < reduc) {
          k.done = 1;
          continue;
        }
        if (!BICG) k.cof[4] = k.cof[0];
      }
      all = false;
      if (BICG) {
        k.cof[1] = 0.0;
        k.cof[4] = t[NC + q];
        k.cof[6] = k.cof[4] * k.cof[5] / (k.cof[2] * k.cof[3] + SMALL);
        k.cof[3] = k.cof[4];
      }
    }
  done_store(slot, all);
}

static int fl_pgrid(int n) { return red_grid(n); }

// ---------------------------------------------------------------- one-launch sweeps
__global__ __launch_bounds__(BS) void k_fl_mark(size_t cnt, double *out, int *ticket, const FlKS *ks, int ncmp) {
  if (fl_all_done(ks, ncmp)) return;
  unsigned long long *o = (unsigned long long *)out;
  for (size_t i = blockIdx.x * (size_t)BS + threadIdx.x; i < cnt; i += (size_t)gridDim.x * BS) o[i] = kSweepMark;
  if (blockIdx.x == 0 && threadIdx.x == 0) *ticket = 0;
}

// preconditioner (solv_m.f90:224-250) for one row: the lower entries in
// column order
struct FlPcRow {
  const int *ia, *ja, *kii, *klo, *tpos, *order;
  const double *a;
  double *pc;
  int r, k, nl;
  double s;
  int j[kSweepSlots];
  double a1[kSweepSlots], a2[kSweepSlots];
  __device__ void start(int pos) {
    r = order[pos];
    const int lo = ia[r];
    nl = klo[r] - lo;
    s = a[kii[r]];
    k = 0;
#pragma unroll
    for (int t = 0; t < kSweepSlots; ++t) {
      j[t] = 0;
      a1[t] = a2[t] = 0.0;
      if (t < nl) {
        j[t] = ja[lo + t];
        a1[t] = a[lo + t];
        a2[t] = a[tpos[lo + t]];
      }
    }
  }
  __device__ bool advance() {
    unsigned long long v[kSweepSlots];
#pragma unroll
    for (int t = 0; t < kSweepSlots; ++t)
      if (t >= k && t < nl) v[t] = ld_agent(pc + j[t]);
#pragma unroll
    for (int t = 0; t < kSweepSlots; ++t) {
      if (t < k || t >= nl) continue;
      if (v[t] == kSweepMark) break;
      s = s - a1[t] * __longlong_as_double((long long)v[t]) * a2[t];
      k = t + 1;
    }
    if (k < nl) return false;
    st_agent(pc + r, 1.0 / (s + SMALL));
    return true;
  }
};

// direct_solve for NC right-hand sides: forward (solv_m.f90:255-268) writes
// out from src = b; backward (:270-286) scales src = the forward result and
// writes out from the upper entries, last column first
template <bool FWD, int NC>
struct FlSweepRow {
  const int *ia, *ja, *klo, *kup, *order;
  const double *a, *pc, *src;
  double *out;
  int n, r, k, nl;
  double s[NC];
  int j[kSweepSlots];
  double av[kSweepSlots];
  __device__ void start(int pos) {
    r = order[pos];
    int first, step;
    if (FWD) {
      first = ia[r];
      nl = klo[r] - first;
      step = 1;
    } else {
      first = ia[r + 1] - 1;
      nl = first - kup[r] + 1;
      step = -1;
    }
    k = 0;
#pragma unroll
    for (int t = 0; t < kSweepSlots; ++t) {
      j[t] = 0;
      av[t] = 0.0;
      if (t < nl) {
        j[t] = ja[first + step * t];
        av[t] = a[first + step * t];
      }
    }
    if (FWD) {
#pragma unroll
      for (int q = 0; q < NC; ++q) s[q] = src[(size_t)q * n + r];
    } else {
      const double cof = 1.0 / (pc[r] + SMALL);
#pragma unroll
      for (int q = 0; q < NC; ++q) s[q] = cof * src[(size_t)q * n + r];
    }
  }
  __device__ bool advance() {
    unsigned long long v[kSweepSlots][NC];
#pragma unroll
    for (int t = 0; t < kSweepSlots; ++t)
      if (t >= k && t < nl)
#pragma unroll
        for (int q = 0; q < NC; ++q) v[t][q] = ld_agent(out + (size_t)q * n + j[t]);
#pragma unroll
    for (int t = 0; t < kSweepSlots; ++t) {
      if (t < k || t >= nl) continue;
      bool ready = true;
#pragma unroll
      for (int q = 0; q < NC; ++q) ready = ready && v[t][q] != kSweepMark;
      if (!ready) break;
#pragma unroll
      for (int q = 0; q < NC; ++q) s[q] = s[q] - av[t] * __longlong_as_double((long long)v[t][q]);
      k = t + 1;
    }
    if (k < nl) return false;
    const double cc = pc[r];
#pragma unroll
    for (int q = 0; q < NC; ++q) st_agent(out + (size_t)q * n + r, s[q] * cc);
    return true;
  }
};

__global__ __launch_bounds__(BS) void k_fl_pc_sf(int n, const int *__restrict__ order, const int *__restrict__ ia,
                                                 const int *__restrict__ ja, const int *__restrict__ kii,
                                                 const int *__restrict__ klo, const int *__restrict__ tpos,
                                                 const double *__restrict__ a, double *pc, int *ticket, int *err) {
  FlPcRow row;
  row.ia = ia; row.ja = ja; row.kii = kii; row.klo = klo; row.tpos = tpos; row.order = order; row.a = a; row.pc = pc;
  row.r = 0; row.k = 0; row.nl = 0; row.s = 0.0;
  sweep_chunks(n, ticket, err, row);
}

template <bool FWD, int NC>
__global__ __launch_bounds__(BS) void k_fl_sweep_sf(int n, const int *__restrict__ order, const int *__restrict__ ia,
                                                    const int *__restrict__ ja, const int *__restrict__ klo,
                                                    const int *__restrict__ kup, const double *__restrict__ a,
                                                    const double *__restrict__ pc, const double *__restrict__ src,
                                                    double *out, int *ticket, int *err, const FlKS *ks) {
  if (fl_all_done(ks, NC)) return;
  FlSweepRow<FWD, NC> row;
  row.ia = ia; row.ja = ja; row.klo = klo; row.kup = kup; row.order = order; row.a = a; row.pc = pc; row.src = src;
  row.out = out; row.n = n; row.r = 0; row.k = 0; row.nl = 0;
  sweep_chunks(n, ticket, err, row);
}

// ---------------------------------------------------------------- host
// The sweeps' pattern: lower entries in column order, upper entries from the
// row's last column down, as direct_solve takes them.
static SweepGraph fl_sweep_graph(int n, const std::vector<int> &ia, const std::vector<int> &ja,
                                 const std::vector<int> &klo, const std::vector<int> &kup,
                                 const std::vector<int> &tpos) {
  SweepGraph g;
  g.n = n;
  g.row.resize(n);
  for (int r = 0; r < n; ++r) g.row[r] = r;
  g.lptr.assign(n + 1, 0);
  g.uptr.assign(n + 1, 0);
  bool sorted = true;
  for (int r = 0; r < n; ++r) {
    g.lptr[r + 1] = g.lptr[r] + klo[r] - ia[r];
    g.uptr[r + 1] = g.uptr[r] + ia[r + 1] - kup[r];
    for (int k = ia[r] + 1; k < ia[r + 1]; ++k) sorted = sorted && ja[k - 1] < ja[k];
  }
  // every lower entry has its transpose (checked with tpos); in sorted rows
  // with as many upper entries these are all of them
  g.symmetric = sorted && g.lptr[n] == g.uptr[n];
  g.lcol.reserve(g.lptr[n]);
  g.lval.reserve(g.lptr[n]);
  g.tval.reserve(g.lptr[n]);
  g.ucol.reserve(g.uptr[n]);
  g.uval.reserve(g.uptr[n]);
  for (int r = 0; r < n; ++r) {
    for (int k = ia[r]; k < klo[r]; ++k) {
      g.lcol.push_back(ja[k]);
      g.lval.push_back(k);
      g.tval.push_back(tpos[k]);
    }
    for (int k = ia[r + 1] - 1; k >= kup[r]; --k) {
      g.ucol.push_back(ja[k]);
      g.uval.push_back(k);
    }
  }
  return g;
}

static int fl_parts_setup(FlCtx &c) {
  sweep_exec_free(c.sw);
  const SweepGraph g = fl_sweep_graph(c.n, c.h_ia, c.h_ja, c.h_klo, c.h_kup, c.h_tpos);
  SweepPlan p;
  // no plan, a slower one, or no room for its tables: the rows are taken in
  // level order in chunks (fl_parts_on)
  if (!sweep_plan(g, c.part_rows, p, c.positions).empty()) return 0;
  if (p.chunks_faster() && c.parts < 2) return 0;
  c.sw.n_cu = c.n_cu;
  return sweep_exec_build(c.sw, p, c.stream);
}

static int fl_levels(const std::vector<int> &ia, const std::vector<int> &ja, int n, bool fwd,
                     std::vector<int> &ptr, std::vector<int> &rows) {
  std::vector<int> lev(n, 0);
  int nl = 0;
  for (int s = 0; s < n; ++s) {
    const int i = fwd ? s : n - 1 - s;
    int l = 0;
    for (int k = ia[i]; k < ia[i + 1]; ++k) {
      const int j = ja[k];
      if (fwd ? j < i : j > i) l = std::max(l, lev[j] + 1);
    }
    lev[i] = l;
    nl = std::max(nl, l + 1);
  }
  ptr.assign(nl + 1, 0);
  for (int i = 0; i < n; ++i) ptr[lev[i] + 1]++;
  for (int l = 0; l < nl; ++l) ptr[l + 1] += ptr[l];
  rows.assign(n, 0);
  std::vector<int> pos(ptr.begin(), ptr.end() - 1);
  for (int i = 0; i < n; ++i) rows[pos[lev[i]]++] = i;
  return 0;
}

static int fl_sweep_grid(const FlCtx &c) {
  return std::max(1, std::min((c.n + BS - 1) / BS, c.sweep_blocks > 0 ? c.sweep_blocks : c.n_cu));
}
static int fl_mark_grid(size_t cnt) { return (int)std::max<size_t>(1, std::min<size_t>((cnt + BS - 1) / BS, 4096)); }

static bool fl_parts_on(const FlCtx &c) { return c.one_launch && c.parts && c.sw.built; }

static int fl_precond(FlCtx &c, const double *a) {
  if (fl_parts_on(c)) {
    const int rc = sweep_pack(c.sw, c.stream, a, a);
    return rc ? rc : sweep_factor(c.sw, c.stream, SWEEP_FL, a, c.kii, c.pc, nullptr, c.sweep_int + 3);
  }
  if (c.one_launch) {
    k_fl_mark<<<fl_mark_grid(c.n), BS, 0, c.stream>>>(c.n, c.pc, c.sweep_int + 2, nullptr, 1);
    k_fl_pc_sf<<<fl_sweep_grid(c), BS, 0, c.stream>>>(c.n, c.lf_rows, c.ia, c.ja, c.kii, c.klo, c.tpos, a, c.pc,
                                                       c.sweep_int + 2, c.sweep_int + 3);
    FVK_HIP(hipGetLastError());
    return 0;
  }
  for (size_t l = 0; l + 1 < c.lf_ptr.size(); ++l) {
    const int cnt = c.lf_ptr[l + 1] - c.lf_ptr[l];
    k_fl_pc_level<<<grid_for(cnt), BS, 0, c.stream>>>(c.lf_rows + c.lf_ptr[l], cnt, c.ia, c.ja, c.kii, c.tpos, a,
                                                       c.pc);
  }
  FVK_HIP(hipGetLastError());
  return 0;
}

// x = M^-1 b (direct_solve), t: scratch
static int fl_direct(FlCtx &c, int ncmp, const double *a, const double *b, double *t, double *x, const FlKS *ks) {
  if (fl_parts_on(c)) {
    SweepGate G;
    if (ks) G = SweepGate{&ks->done, (int)(sizeof(FlKS) / sizeof(int)), ncmp};
    return sweep_apply(c.sw, c.stream, ncmp, b, x, G, c.sweep_int + 3);
  }
  if (c.one_launch) {
    const size_t cnt = (size_t)ncmp * c.n;
    const int G = fl_sweep_grid(c);
    k_fl_mark<<<fl_mark_grid(cnt), BS, 0, c.stream>>>(cnt, t, c.sweep_int, ks, ncmp);
#define FWD(C) k_fl_sweep_sf<true, C><<<G, BS, 0, c.stream>>>(c.n, c.lf_rows, c.ia, c.ja, c.klo, c.kup, a, c.pc, b, \
                                                              t, c.sweep_int, c.sweep_int + 3, ks)
#define BWD(C) k_fl_sweep_sf<false, C><<<G, BS, 0, c.stream>>>(c.n, c.lb_rows, c.ia, c.ja, c.klo, c.kup, a, c.pc, t, \
                                                               x, c.sweep_int + 1, c.sweep_int + 3, ks)
    if (ncmp == 1) FWD(1); else if (ncmp == 2) FWD(2); else FWD(3);
    k_fl_mark<<<fl_mark_grid(cnt), BS, 0, c.stream>>>(cnt, x, c.sweep_int + 1, ks, ncmp);
    if (ncmp == 1) BWD(1); else if (ncmp == 2) BWD(2); else BWD(3);
#undef FWD
#undef BWD
    FVK_HIP(hipGetLastError());
    return 0;
  }
  for (size_t l = 0; l + 1 < c.lf_ptr.size(); ++l) {
    const int cnt = c.lf_ptr[l + 1] - c.lf_ptr[l];
    k_fl_fwd_level<<<grid_for(cnt), BS, 0, c.stream>>>(c.lf_rows + c.lf_ptr[l], cnt, c.n, ncmp, c.ia, c.ja, a, c.pc,
                                                        b, t, ks);
  }
  for (size_t l = 0; l + 1 < c.lb_ptr.size(); ++l) {
    const int cnt = c.lb_ptr[l + 1] - c.lb_ptr[l];
    k_fl_bwd_level<<<grid_for(cnt), BS, 0, c.stream>>>(c.lb_rows + c.lb_ptr[l], cnt, c.n, ncmp, c.ia, c.ja, a, c.pc,
                                                        t, x, ks);
  }
  FVK_HIP(hipGetLastError());
  return 0;
}

template <int NC, int WS>
static int fl_solve_run(FlCtx &c, const FlMat &M, bool bicg, const double *a, double *phi, double *res, int n_iter,
                        double reduc) {
  const int n = c.n, P = fl_pgrid(n), G = grid_for(n);
  double *w1 = wkv(c, 0), *w2 = wkv(c, 1), *w3 = wkv(c, 2), *w4 = wkv(c, 3), *w5 = wkv(c, 4), *wt = wkv(c, 5);
  double *pa = c.part, *pb = c.part + (size_t)6 * RG;
  auto end = [&](int first, const double *part) {
    const DoneSlot w = c.watch.next();
    if (bicg) k_fl_end<NC, true><<<1, RB, 0, c.stream>>>(first, P, part, c.ks, reduc, w);
    else k_fl_end<NC, false><<<1, RB, 0, c.stream>>>(first, P, part, c.ks, reduc, w);
  };
  k_fl_init<NC, WS><<<P, RB, 0, c.stream>>>(M, phi, res, w1, w2, bicg ? w3 : nullptr, pa);
  end(1, pa);
  int rc = fl_precond(c, a);
  if (rc) return rc;
  for (int it = 0; it < n_iter; ++it) {
    if (!bicg) {
      double *po = it & 1 ? w5 : w2, *pn = it & 1 ? w2 : w5;
      if ((rc = fl_direct(c, NC, a, w1, wt, w3, c.ks))) return rc;
      k_fl_dot<NC><<<P, RB, 0, c.stream>>>(n, w1, w3, c.ks, pa);
      k_fl_cg_pq<NC, WS><<<P, RB, 0, c.stream>>>(M, w3, po, pn, w4, pa, P, c.ks, pb);
      k_fl_cg_upd<NC><<<P, RB, 0, c.stream>>>(n, phi, pn, w1, w4, pb, P, c.ks, pa);
      end(0, pa);
    } else {
      k_fl_bi_dir<NC><<<G, BS, 0, c.stream>>>(n, w2, w1, w3, c.ks);
      if ((rc = fl_direct(c, NC, a, w2, wt, w5, c.ks))) return rc;
      k_fl_bi_mv<NC, WS, false><<<P, RB, 0, c.stream>>>(M, w5, w3, res, c.ks, pb);
      k_fl_bi_upd1<NC><<<P, RB, 0, c.stream>>>(n, phi, w5, w1, w3, pb, P, c.ks);
      if ((rc = fl_direct(c, NC, a, w1, wt, w5, c.ks))) return rc;
      k_fl_bi_mv<NC, WS, true><<<P, RB, 0, c.stream>>>(M, w5, w4, w1, c.ks, pa);
      k_fl_bi_upd2<NC><<<P, RB, 0, c.stream>>>(n, phi, w5, w1, w4, res, pa, P, c.ks, pb);
      end(0, pb);
    }
    // the iteration before this one, while this one runs
    bool done = false;
    if (it > 0 && it + 1 < n_iter) FVK_HIP(c.watch.wait(c.stream, c.watch.tag - 1, done));
    if (done) break;
  }
  FVK_HIP(hipGetLastError());
  return 0;
}

// lin_eqns_solver (solv_m.f90:10-30) for ncmp right-hand sides sharing the
// matrix a (device, CSR of the context): phi and res (the right-hand side
// in, the initial residual out) component-major on the device; norms to
// ks[c].norm.  isol 1: cg_solver, 2: bicg_solver.
static int fl_solve(FlCtx &c, int isol, int ncmp, const double *a, double *phi, double *res, int n_iter,
                    double reduc) {
  const FlMat M{c.n, c.ia, c.ja, c.ecol, a, c.eval};
  if (c.ew) k_fl_slots<<<grid_for(c.n), BS, 0, c.stream>>>(M, c.ew, nullptr, c.eval);
  const bool bi = isol == 2;
#define RUN(W)                                                                                    \
  (ncmp == 1   ? fl_solve_run<1, W>(c, M, bi, a, phi, res, n_iter, reduc)                         \
   : ncmp == 2 ? fl_solve_run<2, W>(c, M, bi, a, phi, res, n_iter, reduc)                         \
               : fl_solve_run<3, W>(c, M, bi, a, phi, res, n_iter, reduc))
  return c.ew == 4 ? RUN(4) : c.ew == 5 ? RUN(5) : c.ew == 7 ? RUN(7) : c.ew == 8 ? RUN(8) : RUN(0);
#undef RUN
}

// ---------------------------------------------------------------- SIMPLE
struct FlCfg {
  double cc, cd, urf_u, urf_p, bl_c;
  int n_iter_u, n_iter_p;
  double reduc_u, reduc_p;
};

struct FlFlow {
  FlCtx *c = nullptr;
  FlCfg cfg{};
  std::vector<void *> owned;
  double *u = nullptr, *ub = nullptr, *ug = nullptr;   // velocity: cells, boundary, gradient
  double *p = nullptr, *pb = nullptr, *pg = nullptr;   // pressure
  double *q = nullptr, *qb = nullptr, *qg = nullptr;   // pressure correction
  double *rhs = nullptr, *diag = nullptr, *val = nullptr, *spd = nullptr;
  double *cc = nullptr, *ccb = nullptr, *cd = nullptr, *cdb = nullptr;
  double *fa = nullptr, *fb = nullptr, *fd = nullptr, *fcc = nullptr, *fdc = nullptr;  // face terms
  int *bfl = nullptr;          // boundary faces
  int n_bf = 0;
  double res0[4] = {0, 0, 0, 0};
};

template <class T>
static int ff_alloc(FlFlow &F, T **p, size_t n) {
  void *q = nullptr;
  FVK_HIP(hipMalloc(&q, (n ? n : 1) * sizeof(T)));
  F.owned.push_back(q);
  FVK_HIP(hipMemsetAsync(q, 0, (n ? n : 1) * sizeof(T), F.c->stream));
  FVK_HIP(hipStreamSynchronize(F.c->stream));
  *p = (T *)q;
  return 0;
}

// boundary type ranges (transport_m.f90:11-14)
__device__ __forceinline__ bool fl_is(int ty, int lo) { return ty >= lo && ty <= lo + 9; }

__global__ __launch_bounds__(BS) void k_fl_fill(size_t n, double *a, double v) {
  for (size_t i = blockIdx.x * (size_t)BS + threadIdx.x; i < n; i += (size_t)gridDim.x * BS) a[i] = v;
}

// ns_source (transport_m.f90:726-752): rhs = 0 + (-grad p) vol
__global__ __launch_bounds__(BS) void k_fl_source(int n, int nd, const double *__restrict__ pg,
                                                  const double *__restrict__ vol, double *rhs) {
  const int i = blockIdx.x * BS + threadIdx.x;
  if (i >= n) return;
  for (int d = 0; d < nd; ++d) rhs[(size_t)d * n + i] = 0.0 + (-pg[(size_t)d * n + i]) * vol[i];
}

struct FlGeo {
  int n, nf, nb, nd;
  const int *j1, *jn, *btag, *kij, *kji;
  const double *xvc, *xfc, *nrm, *area, *xpc, *lpn, *wfp;
};

// construct_pde face terms (transport_m.f90:97-297)
__global__ __launch_bounds__(BS) void k_fl_pde_face(FlGeo g, double bl_c, const double *__restrict__ u,
                                                    double *ub, const double *__restrict__ ug,
                                                    const double *__restrict__ spd, const double *__restrict__ cc,
                                                    const double *__restrict__ ccb, const double *__restrict__ cd,
                                                    const double *__restrict__ cdb, double *val, double *fa,
                                                    double *fb, double *fd, double *fcc, double *fdc) {
  const int f = xcd_block() * BS + threadIdx.x;
  if (f >= g.nf) return;
  const int n = g.n, nf = g.nf, nd = g.nd, p = g.j1[f], q = g.jn[f];
  const double ar = g.area[f];
  double nv[3] = {0, 0, 0};
  for (int d = 0; d < nd; ++d) nv[d] = g.nrm[(size_t)d * nf + f];
  if (q >= 0) {
    const double w = g.wfp[f], wn = 1.0 - w;
    double del[3] = {0, 0, 0}, dl = 0.0;
    for (int d = 0; d < nd; ++d) del[d] = g.xvc[(size_t)d * n + q] - g.xvc[(size_t)d * n + p];
    for (int d = 0; d < nd; ++d) dl = dl + del[d] * del[d];
    const double dm = sqrt(dl) + SMALL;
    for (int d = 0; d < nd; ++d) del[d] = nv[d] - del[d] / dm;
    double fg[3][3];  // fg[d][c] = grad(d, c)
    for (int c = 0; c < nd; ++c)
      for (int d = 0; d < nd; ++d)
        fg[d][c] = w * ug[(size_t)(c * nd + d) * n + q] + wn * ug[(size_t)(c * nd + d) * n + p];
    double dx[3];
    for (int d = 0; d < nd; ++d)
      dx[d] = g.xfc[(size_t)d * nf + f] - (w * g.xvc[(size_t)d * n + q] + wn * g.xvc[(size_t)d * n + p]);
    double fphi[3];
    for (int c = 0; c < nd; ++c) {
      double s = 0.0;
      for (int d = 0; d < nd; ++d) s = s + fg[d][c] * dx[d];
      fphi[c] = w * u[(size_t)c * n + q] + wn * u[(size_t)c * n + p] + s;
    }
    const double fc = w * cc[q] + wn * cc[p];
    const double fdd = w * cd[q] + wn * cd[p];
    const double cv = fc * ar * spd[f];
    const double dv = fdd * ar / g.lpn[f];
    const double c_ij = fmin(cv, 0.0), c_ji = -fmax(cv, 0.0), d_ij = -dv;
    for (int c = 0; c < nd; ++c) {
      const double imp = cv > 0.0 ? u[(size_t)c * n + p] : u[(size_t)c * n + q];
      const double c_cor = bl_c * cv * (imp - fphi[c]);
      double dc = 0.0;
      for (int d = 0; d < nd; ++d) dc = dc + fg[d][c] * del[d];
      dc = dc * fdd * ar;
      double de = 0.0;
      for (int d = 0; d < nd; ++d) de = de + fg[c][d] * nv[d];
      de = de * fdd * ar;
      dc = dc + de;
      fcc[(size_t)c * nf + f] = c_cor;
      fdc[(size_t)c * nf + f] = dc;
    }
    val[g.kij[f]] = 0.0 + c_ij + d_ij;
    val[g.kji[f]] = 0.0 + c_ji + d_ij;
    fa[f] = c_ij;
    fb[f] = c_ji;
    fd[f] = d_ij;
  } else {
    const int b = -q - 1, ty = g.btag[b];
    double fg[3][3];
    for (int c = 0; c < nd; ++c)
      for (int d = 0; d < nd; ++d) fg[d][c] = ug[(size_t)(c * nd + d) * n + p];
    double fphi[3], vphi[3];
    for (int c = 0; c < nd; ++c) {
      fphi[c] = ub[(size_t)c * g.nb + b];
      vphi[c] = u[(size_t)c * n + p];
    }
    const double fc = ccb[b], fdd = cdb[b];
    const double cv = fc * ar * spd[f];
    const double dv = fdd * ar / g.lpn[f];
    double c_ij = fmin(cv, 0.0), d_ij = -dv;
    double vn = 0.0;
    for (int d = 0; d < nd; ++d) vn = vn + vphi[d] * nv[d];
    double dexp[3];
    for (int c = 0; c < nd; ++c) {
      if (fl_is(ty, 30)) {
        dexp[c] = fphi[c] - (vphi[c] - nv[c] * vn);
        dexp[c] = dexp[c] / g.lpn[f];
      } else if (fl_is(ty, 40)) {
        dexp[c] = 2.0 * (0.0 - nv[c] * vn);
        dexp[c] = dexp[c] / g.lpn[f];
      } else {
        double s = 0.0;
        for (int d = 0; d < nd; ++d) s = s + (fg[c][d] + fg[d][c]) * nv[d];
        dexp[c] = s;
      }
    }
    double dcor[3];
    for (int c = 0; c < nd; ++c) dcor[c] = fdd * ar * dexp[c] - dv * (fphi[c] - vphi[c]);
    if (fl_is(ty, 20)) {
      for (int c = 0; c < nd; ++c) fphi[c] = vphi[c];
      c_ij = 0.0;
      d_ij = 0.0;
    } else if (fl_is(ty, 40)) {
      for (int c = 0; c < nd; ++c) fphi[c] = vphi[c] - nv[c] * vn;
    }
    for (int c = 0; c < nd; ++c) {
      ub[(size_t)c * g.nb + b] = fphi[c];
      fcc[(size_t)c * nf + f] = fphi[c];
      fdc[(size_t)c * nf + f] = dcor[c];
    }
    fa[f] = c_ij;
    fd[f] = d_ij;
  }
}

// construct_pde cell part: diagonal and right-hand side gathered over the
// cell's faces (ascending), then under-relaxation (transport_m.f90:300-347)
__global__ __launch_bounds__(BS) void k_fl_pde_cell(int n, int nf, int nd, const int *__restrict__ cptr,
                                                    const int *__restrict__ cfl, const int *__restrict__ j1,
                                                    const int *__restrict__ jn, const int *__restrict__ kii,
                                                    const double *__restrict__ fa, const double *__restrict__ fb,
                                                    const double *__restrict__ fd, const double *__restrict__ fcc,
                                                    const double *__restrict__ fdc, const double *__restrict__ u,
                                                    double urf, double *val, double *rhs, double *diag) {
  const int i = xcd_block() * BS + threadIdx.x;
  if (i >= n) return;
  double v = 0.0, r[3] = {0, 0, 0};
  for (int c = 0; c < nd; ++c) r[c] = rhs[(size_t)c * n + i];
  for (int k = cptr[i]; k < cptr[i + 1]; ++k) {
    const int f = cfl[k];
    if (jn[f] < 0) {
      v = v - fa[f] - fd[f];
      const double cd = fa[f] + fd[f];
      for (int c = 0; c < nd; ++c) r[c] = r[c] - cd * fcc[(size_t)c * nf + f] + fdc[(size_t)c * nf + f];
    } else if (j1[f] == i) {
      v = v - fa[f] - fd[f];
      for (int c = 0; c < nd; ++c) r[c] = r[c] + fcc[(size_t)c * nf + f] + fdc[(size_t)c * nf + f];
    } else {
      v = v - fb[f] - fd[f];
      for (int c = 0; c < nd; ++c) r[c] = r[c] - fcc[(size_t)c * nf + f] - fdc[(size_t)c * nf + f];
    }
  }
  const double urfr = 1.0 / urf;
  v = v * urfr;
  for (int c = 0; c < nd; ++c) rhs[(size_t)c * n + i] = r[c] + (1.0 - urf) * v * u[(size_t)c * n + i];
  val[kii[i]] = v;
  diag[i] = 1.0 / v;
}

// construct_pp face terms (transport_m.f90:466-570), first pass
__global__ __launch_bounds__(BS) void k_fl_pp_face(FlGeo g, const double *__restrict__ u, const double *__restrict__ ub,
                                                   const double *__restrict__ ug, const double *__restrict__ pr,
                                                   const double *__restrict__ pg, const double *__restrict__ cc,
                                                   const double *__restrict__ ccb, const double *__restrict__ diag,
                                                   double *spd, double *val, double *fa, double *fd, double *fdc) {
  const int f = xcd_block() * BS + threadIdx.x;
  if (f >= g.nf) return;
  const int n = g.n, nf = g.nf, nd = g.nd, p = g.j1[f], q = g.jn[f];
  const double ar = g.area[f];
  double nv[3] = {0, 0, 0};
  for (int d = 0; d < nd; ++d) nv[d] = g.nrm[(size_t)d * nf + f];
  if (q >= 0) {
    const double w = g.wfp[f], wn = 1.0 - w;
    double dx[3];
    for (int d = 0; d < nd; ++d)
      dx[d] = g.xfc[(size_t)d * nf + f] - (w * g.xvc[(size_t)d * n + q] + wn * g.xvc[(size_t)d * n + p]);
    double fv[3];
    for (int c = 0; c < nd; ++c) {
      double s = 0.0;
      for (int d = 0; d < nd; ++d)
        s = s + (w * ug[(size_t)(c * nd + d) * n + q] + wn * ug[(size_t)(c * nd + d) * n + p]) * dx[d];
      fv[c] = w * u[(size_t)c * n + q] + wn * u[(size_t)c * n + p] + s;
    }
    double sp = 0.0;
    for (int d = 0; d < nd; ++d) sp = sp + fv[d] * nv[d];
    spd[f] = sp;
    const double fc = w * cc[q] + wn * cc[p];
    const double fapr = w * diag[q] + wn * diag[p];
    const double d_ij = -(fc * fapr * (ar * ar));
    const double cv = -(fc * ar * sp);
    double t = 0.0;
    for (int d = 0; d < nd; ++d)
      t = t + (w * pg[(size_t)d * n + q] + wn * pg[(size_t)d * n + p]) *
                  (g.xvc[(size_t)d * n + q] - g.xvc[(size_t)d * n + p]);
    double dcor = pr[q] - pr[p];
    dcor = dcor - t;
    dcor = -(dcor * d_ij);
    val[g.kij[f]] = 0.0 + d_ij;
    val[g.kji[f]] = 0.0 + d_ij;
    fa[f] = cv;
    fd[f] = d_ij;
    fdc[f] = dcor;
  } else {
    const int b = -q - 1;
    double sp = 0.0;
    for (int d = 0; d < nd; ++d) sp = sp + ub[(size_t)d * g.nb + b] * nv[d];
    double cv = -(ccb[b] * ar * sp);
    if (fl_is(g.btag[b], 20)) {
      if (sp < 0.0) sp = 0.0;
      cv = 0.0;
    }
    spd[f] = sp;
    fa[f] = cv;
  }
}

// flux_out_corr (transport_m.f90:350-425): inlet and outlet mass fluxes
__global__ __launch_bounds__(RB) void k_fl_inout(int nbf, const int *__restrict__ bfl, const int *__restrict__ jn,
                                                 const int *__restrict__ btag, const double *__restrict__ ccb,
                                                 const double *__restrict__ area, const double *__restrict__ spd,
                                                 double *part) {
  double v[2] = {0.0, 0.0};
  for (int t = blockIdx.x * RB + threadIdx.x; t < nbf; t += gridDim.x * RB) {
    const int f = bfl[t], b = -jn[f] - 1, ty = btag[b];
    const double c = ccb[b] * area[f] * spd[f];
    if (fl_is(ty, 10)) v[0] += c;
    else if (fl_is(ty, 20)) v[1] += c;
  }
  rblock_sum<2, RB>(v);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = v[0];
    part[RG + blockIdx.x] = v[1];
  }
}

__global__ __launch_bounds__(RB) void k_fl_crat(int P, const double *part, double *scal) {
  double t[2];
  load_totals<2, RB>(part, P, t);
  const double ci = t[0], co = t[1];
  if (threadIdx.x == 0) {
    double r = ci / (co + SMALL);
    r = fabs(r);
    scal[0] = fmin(1000.0, r);
  }
}

// outlet fluxes scaled by c_rat (transport_m.f90:599-627)
__global__ __launch_bounds__(BS) void k_fl_outlet(int nbf, const int *__restrict__ bfl, const int *__restrict__ jn,
                                                  const int *__restrict__ btag, const double *__restrict__ scal,
                                                  double *spd) {
  const int t = blockIdx.x * BS + threadIdx.x;
  if (t >= nbf) return;
  const int f = bfl[t], b = -jn[f] - 1;
  if (fl_is(btag[b], 20)) spd[f] = spd[f] * scal[0];
}

// construct_pp cell part: diagonal, right-hand side (first pass over the
// faces, then the outlet faces' corrected fluxes)
__global__ __launch_bounds__(BS) void k_fl_pp_cell(int n, int nb, const int *__restrict__ cptr,
                                                   const int *__restrict__ cfl, const int *__restrict__ j1,
                                                   const int *__restrict__ jn, const int *__restrict__ kii,
                                                   const int *__restrict__ btag, const double *__restrict__ ccb,
                                                   const double *__restrict__ area, const double *__restrict__ spd,
                                                   const double *__restrict__ fa, const double *__restrict__ fd,
                                                   const double *__restrict__ fdc, double *val, double *rhs) {
  const int i = xcd_block() * BS + threadIdx.x;
  if (i >= n) return;
  double v = 0.0, r = 0.0;
  for (int k = cptr[i]; k < cptr[i + 1]; ++k) {
    const int f = cfl[k];
    if (jn[f] < 0) {
      r = r + fa[f];
    } else if (j1[f] == i) {
      v = v - fd[f];
      r = r + fa[f] + fdc[f];
    } else {
      v = v - fd[f];
      r = r - fa[f] - fdc[f];
    }
  }
  for (int k = cptr[i]; k < cptr[i + 1]; ++k) {
    const int f = cfl[k];
    if (jn[f] >= 0) continue;
    const int b = -jn[f] - 1;
    if (!fl_is(btag[b], 20)) continue;
    r = r + -(ccb[b] * area[f] * spd[f]);
  }
  val[kii[i]] = v;
  rhs[i] = r;
}

// ns_correction (transport_m.f90:757-800); the serial build keeps the
// reference pressure at its initial zero (blk is 1 there)
__global__ __launch_bounds__(BS) void k_fl_correct(int n, int nd, const double *__restrict__ qg,
                                                   const double *__restrict__ vol, const double *__restrict__ diag,
                                                   const double *__restrict__ q, double ref, double urf, double *u,
                                                   double *p) {
  const int i = blockIdx.x * BS + threadIdx.x;
  if (i >= n) return;
  for (int d = 0; d < nd; ++d) {
    double dv = -qg[(size_t)d * n + i];
    dv = dv * vol[i] * diag[i];
    u[(size_t)d * n + i] = u[(size_t)d * n + i] + dv;
  }
  const double dp = (q[i] - ref) * urf;
  p[i] = p[i] + dp;
}

static FlGeo fl_geo(const FlCtx &c) {
  FlGeo g;
  g.n = c.n; g.nf = c.nf; g.nb = c.nb; g.nd = c.nd;
  g.j1 = c.j1; g.jn = c.jn; g.btag = c.btag; g.kij = c.kij; g.kji = c.kji;
  g.xvc = c.xvc; g.xfc = c.xfc; g.nrm = c.nrm; g.area = c.area; g.xpc = c.xpc; g.lpn = c.lpn; g.wfp = c.wfp;
  return g;
}

int fl_grad(FlCtx &c, int ncmp, const double *phi, double *phib, double *g, int neu, const int *bfl, int n_bf) {
  k_fl_grad<<<grid_for(c.n), BS, 0, c.stream>>>(c.n, c.nf, c.nb, c.nd, ncmp, c.cptr, c.cfl, c.j1, c.jn, c.xvc, c.xfc,
                                                 c.ls, phi, phib, neu, g);
  if (neu && n_bf)
    k_fl_grad_bnd<<<grid_for(n_bf), BS, 0, c.stream>>>(n_bf, bfl, c.n, c.nf, c.nb, c.nd, ncmp, c.j1, c.jn, c.xvc,
                                                        c.xfc, phi, g, phib);
  FVK_HIP(hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------- host set-up
// The cell matrix pattern (1-based CSR) and the Krylov workspace.
struct FlPattern {
  std::vector<int> ia, ja, kii, klo, kup, tpos;
  int widest = 0;  // the most lower or upper entries of a row
};
static int fl_pattern(int n, const int *ngp, const int *ngc, FlPattern &p) {
  const int nnz = ngp[n] - 1;
  if (ngp[0] != 1 || nnz < n) { set_error("bad matrix pattern"); return FVK_ERR_ARG; }
  p.ia.resize(n + 1);
  p.ja.resize(nnz);
  std::vector<int> &ia = p.ia, &ja = p.ja;
  for (int i = 0; i <= n; ++i) {
    ia[i] = ngp[i] - 1;
    if (i && ia[i] < ia[i - 1]) { set_error("bad matrix pattern"); return FVK_ERR_ARG; }
  }
  for (int k = 0; k < nnz; ++k) {
    ja[k] = ngc[k] - 1;
    if (ja[k] < 0 || ja[k] >= n) { set_error("matrix column out of range"); return FVK_ERR_ARG; }
  }
  auto csr_index = [&](int i, int j) {
    for (int k = ia[i]; k < ia[i + 1]; ++k)
      if (ja[k] == j) return k;
    return -1;
  };
  p.kii.resize(n);
  p.klo.resize(n);
  p.kup.resize(n);
  p.tpos.assign(nnz, -1);
  for (int i = 0; i < n; ++i) {
    if ((p.kii[i] = csr_index(i, i)) < 0) { set_error("matrix pattern lacks a diagonal entry"); return FVK_ERR_ARG; }
    int k = ia[i];
    while (k < ia[i + 1] && ja[k] < i) ++k;
    p.klo[i] = k;
    k = ia[i + 1];
    while (k > ia[i] && ja[k - 1] > i) --k;
    p.kup[i] = k;
    p.widest = std::max({p.widest, p.klo[i] - ia[i], ia[i + 1] - p.kup[i]});
    for (int q = ia[i]; q < p.klo[i]; ++q)
      if ((p.tpos[q] = csr_index(ja[q], i)) < 0) { set_error("matrix pattern is not symmetric"); return FVK_ERR_ARG; }
  }
  return 0;
}

static int fl_csr_setup(FlCtx &c, int n, const int *ngp, const int *ngc) {
  c.n = n;
  FlPattern p;
  {
    const int rc = fl_pattern(n, ngp, ngc, p);
    if (rc) return rc;
  }
  c.nnz = (int)p.ja.size();
  const std::vector<int> &ia = p.ia, &ja = p.ja, &kii = p.kii, &klo = p.klo, &kup = p.kup, &tpos = p.tpos;
  const int mx = p.widest;
  c.one_launch = c.narrow = mx <= kSweepSlots;
  c.h_ia = ia;
  c.h_ja = ja;
  c.h_kii = kii;
  c.h_klo = klo;
  c.h_kup = kup;
  c.h_tpos = tpos;
  int rc = 0;
#define A(ptr, cnt_) if (!rc) rc = fl_alloc(c, &ptr, cnt_)
#define U(ptr, vec) if (!rc) rc = fl_up(c, &ptr, vec)
  U(c.ia, ia); U(c.ja, ja); U(c.kii, kii); U(c.klo, klo); U(c.kup, kup); U(c.tpos, tpos);
  A(c.wk, (size_t)6 * 3 * n); A(c.pc, n); A(c.part, (size_t)12 * RG); A(c.ks, 3); A(c.scal, 8);
  A(c.sweep_int, 4);
#undef A
#undef U
  if (rc) return rc;
  FVK_HIP(hipDeviceGetAttribute(&c.n_cu, hipDeviceAttributeMultiprocessorCount, c.device));
  std::vector<int> lrows;
  fl_levels(ia, ja, n, true, c.lf_ptr, lrows);
  if ((rc = fl_up(c, &c.lf_rows, lrows))) return rc;
  fl_levels(ia, ja, n, false, c.lb_ptr, lrows);
  if ((rc = fl_up(c, &c.lb_rows, lrows))) return rc;
  if (c.one_launch) {
    c.parts = 1;
    if ((rc = fl_parts_setup(c))) return rc;
  }
  FVK_HIP(c.watch.init());
  // rows of 4, 5 or 7 entries: triangles, quadrangles, hexahedra; by slots
  // unless half of them would be empty or there is no memory for them
  int w = 0;
  for (int i = 0; i < n; ++i) w = std::max(w, ia[i + 1] - ia[i]);
  w = w <= 4 ? 4 : w == 6 ? 7 : w;
  if (w <= 8 && (size_t)w * n <= 2 * (size_t)c.nnz) {
    void *q = nullptr, *v = nullptr;
    if (hipMalloc(&q, (size_t)w * n * sizeof(int)) == hipSuccess &&
        hipMalloc(&v, (size_t)w * n * sizeof(double)) == hipSuccess) {
      c.owned.push_back(q);
      c.owned.push_back(v);
      c.ecol = (int *)q;
      c.eval = (double *)v;
      c.ew = w;
      k_fl_slots<<<grid_for(n), BS, 0, c.stream>>>(FlMat{n, c.ia, c.ja, nullptr, nullptr, nullptr}, w, c.ecol, nullptr);
      FVK_HIP(hipGetLastError());
      FVK_HIP(hipStreamSynchronize(c.stream));
    } else {
      (void)hipGetLastError();
      if (q) (void)hipFree(q);
    }
  }
  return 0;
}

static int fl_ctx_build(FlCtx &c, int nd, int n_vrt, const double *x3, int nb, const int *btag, int n,
                        const int *evp, const int *evr, int nf, const int *fce_elm, const int *fvp, const int *fvr,
                        const int *ngp, const int *ngc) {
  c.nd = nd; c.n_vrt = n_vrt; c.nb = nb; c.n = n; c.nf = nf;
  {
    const int rc = fl_csr_setup(c, n, ngp, ngc);
    if (rc) return rc;
  }
  // element and face numbering -> 0-based local indices
  std::vector<int> j1(nf), jn(nf);
  for (int f = 0; f < nf; ++f) {
    const int a = fce_elm[2 * f], b = fce_elm[2 * f + 1];
    if (a <= nb || a > nb + n) { set_error("face " + std::to_string(f + 1) + ": owner is not a domain element"); return FVK_ERR_ARG; }
    j1[f] = a - nb - 1;
    if (b > 0) {
      if (b <= nb || b > nb + n) { set_error("face " + std::to_string(f + 1) + ": bad neighbour"); return FVK_ERR_ARG; }
      jn[f] = b - nb - 1;
    } else {
      if (b == 0 || -b > nb) { set_error("face " + std::to_string(f + 1) + ": bad boundary element"); return FVK_ERR_ARG; }
      jn[f] = b;  // -(boundary element), i.e. -(b0 + 1) with b0 0-based
    }
  }
  const std::vector<int> &ia = c.h_ia, &ja = c.h_ja;
  auto csr_index = [&](int i, int j) {
    for (int k = ia[i]; k < ia[i + 1]; ++k)
      if (ja[k] == j) return k;
    return -1;
  };
  std::vector<int> kij(nf, -1), kji(nf, -1);
  for (int f = 0; f < nf; ++f)
    if (jn[f] >= 0) {
      kij[f] = csr_index(j1[f], jn[f]);
      kji[f] = csr_index(jn[f], j1[f]);
      if (kij[f] < 0 || kji[f] < 0) { set_error("matrix pattern lacks a face's entries"); return FVK_ERR_ARG; }
    }
  // cell face lists, ascending
  std::vector<int> cnt(n + 1, 0), cfl;
  for (int f = 0; f < nf; ++f) {
    cnt[j1[f] + 1]++;
    if (jn[f] >= 0) cnt[jn[f] + 1]++;
  }
  for (int i = 0; i < n; ++i) cnt[i + 1] += cnt[i];
  cfl.resize(cnt[n]);
  std::vector<int> fill(cnt.begin(), cnt.end() - 1);
  for (int f = 0; f < nf; ++f) {
    cfl[fill[j1[f]]++] = f;
    if (jn[f] >= 0) cfl[fill[jn[f]]++] = f;
  }
  std::vector<int> evp0(n + 1), evr0(evp[n] - 1), fvp0(nf + 1), fvr0(fvp[nf] - 1);
  for (int i = 0; i <= n; ++i) evp0[i] = evp[i] - 1;
  for (size_t k = 0; k < evr0.size(); ++k) {
    evr0[k] = evr[k] - 1;
    if (evr0[k] < 0 || evr0[k] >= n_vrt) { set_error("element vertex out of range"); return FVK_ERR_ARG; }
  }
  for (int f = 0; f <= nf; ++f) fvp0[f] = fvp[f] - 1;
  for (size_t k = 0; k < fvr0.size(); ++k) {
    fvr0[k] = fvr[k] - 1;
    if (fvr0[k] < 0 || fvr0[k] >= n_vrt) { set_error("face vertex out of range"); return FVK_ERR_ARG; }
  }
  for (int f = 0; f < nf; ++f)
    if (fvp0[f + 1] - fvp0[f] < 2 || (nd == 3 && fvp0[f + 1] - fvp0[f] < 3)) {
      set_error("face with too few vertices");
      return FVK_ERR_ARG;
    }
  c.h_j1 = j1; c.h_jn = jn;
  c.h_btag.assign(btag, btag + nb);
  int rc = 0;
#define A(ptr, cnt_) if (!rc) rc = fl_alloc(c, &ptr, cnt_)
#define U(ptr, vec) if (!rc) rc = fl_up(c, &ptr, vec)
  std::vector<double> xv(x3, x3 + 3 * (size_t)n_vrt);
  double *dxv = nullptr;
  int *devp = nullptr, *devr = nullptr, *dfvp = nullptr, *dfvr = nullptr;
  U(dxv, xv); U(devp, evp0); U(devr, evr0); U(dfvp, fvp0); U(dfvr, fvr0);
  U(c.j1, j1); U(c.jn, jn); U(c.btag, c.h_btag);
  U(c.kij, kij); U(c.kji, kji);
  U(c.cptr, cnt); U(c.cfl, cfl);
  A(c.xvc, (size_t)nd * n); A(c.vol, n); A(c.volr, n); A(c.ls, (size_t)nd * nd * n);
  A(c.xfc, (size_t)nd * nf); A(c.nrm, (size_t)nd * nf); A(c.area, nf); A(c.xpc, (size_t)nd * nf);
  A(c.xnc, (size_t)nd * nf); A(c.lpn, nf); A(c.wfp, nf); A(c.fvol, nf);
#undef A
#undef U
  if (rc) return rc;
  k_fl_centre<<<grid_for(n), BS, 0, c.stream>>>(n, nd, dxv, devp, devr, c.xvc);
  k_fl_face_geom<<<grid_for(nf), BS, 0, c.stream>>>(nf, n, nd, dxv, dfvp, dfvr, c.j1, c.jn, c.xvc, c.xfc, c.nrm,
                                                     c.area, c.xpc, c.xnc, c.lpn, c.wfp, c.fvol);
  k_fl_vol<<<grid_for(n), BS, 0, c.stream>>>(n, c.cptr, c.cfl, c.j1, c.fvol, c.vol, c.volr);
  k_fl_ls<<<grid_for(n), BS, 0, c.stream>>>(n, nf, nd, c.cptr, c.cfl, c.j1, c.jn, c.xvc, c.xfc, c.ls);
  FVK_HIP(hipGetLastError());
  FVK_HIP(hipStreamSynchronize(c.stream));
  return 0;
}

static void fl_ctx_free(FlCtx &c) {
  if (c.stream) hipStreamSynchronize(c.stream);
  for (void *p : c.owned) hipFree(p);
  c.owned.clear();
  sweep_exec_free(c.sw);
  c.io.free();
  c.watch.free();
  if (c.stream) hipStreamDestroy(c.stream);
  c.stream = nullptr;
}

// device (component-major, SoA) <-> Fortran column-major a(ncmp, m)
static int fl_in(FlCtx &c, const double *h, int ncmp, int m, double *d) { return c.io.put(h, ncmp, m, nullptr, d, m); }
static int fl_out(FlCtx &c, const double *d, int ncmp, int m, double *h) { return c.io.get(d, m, ncmp, m, nullptr, h); }

static int ff_build(FlFlow &F) {
  FlCtx &c = *F.c;
  const size_t n = c.n, nb = std::max(c.nb, 1), nf = c.nf, nd = c.nd;
  int rc = 0;
#define A(ptr, cnt_) if (!rc) rc = ff_alloc(F, &ptr, cnt_)
  A(F.u, nd * n); A(F.ub, nd * nb); A(F.ug, nd * nd * n);
  A(F.p, n); A(F.pb, nb); A(F.pg, nd * n);
  A(F.q, n); A(F.qb, nb); A(F.qg, nd * n);
  A(F.rhs, nd * n); A(F.diag, n); A(F.val, (size_t)c.nnz); A(F.spd, nf);
  A(F.cc, n); A(F.ccb, nb); A(F.cd, n); A(F.cdb, nb);
  A(F.fa, nf); A(F.fb, nf); A(F.fd, nf); A(F.fcc, nd * nf); A(F.fdc, nd * nf);
#undef A
  if (rc) return rc;
  std::vector<int> bfl;
  for (int f = 0; f < c.nf; ++f)
    if (c.h_jn[f] < 0) bfl.push_back(f);
  F.n_bf = (int)bfl.size();
  {
    void *q = nullptr;
    FVK_HIP(hipMalloc(&q, std::max<size_t>(bfl.size(), 1) * sizeof(int)));
    F.owned.push_back(q);
    F.bfl = (int *)q;
    if (!bfl.empty()) FVK_HIP(hipMemcpy(F.bfl, bfl.data(), bfl.size() * sizeof(int), hipMemcpyHostToDevice));
  }
  const int g = 1024;
  k_fl_fill<<<g, BS, 0, c.stream>>>(n, F.cc, F.cfg.cc);
  k_fl_fill<<<g, BS, 0, c.stream>>>(nb, F.ccb, F.cfg.cc);
  k_fl_fill<<<g, BS, 0, c.stream>>>(n, F.cd, F.cfg.cd);
  k_fl_fill<<<g, BS, 0, c.stream>>>(nb, F.cdb, F.cfg.cd);
  FVK_HIP(hipGetLastError());
  FVK_HIP(hipStreamSynchronize(c.stream));
  return 0;
}

static void ff_free(FlFlow &F) {
  if (F.c && F.c->stream) hipStreamSynchronize(F.c->stream);
  for (void *p : F.owned) hipFree(p);
  F.owned.clear();
}

// the operators of one outer iteration (navierstokes.f90:518-620)
enum FlField { FL_VEL = 0, FL_PRES = 1, FL_PP = 2 };

static int ff_gradient(FlFlow &F, int which, int neu) {
  FlCtx &c = *F.c;
  if (which == FL_VEL) return fl_grad(c, c.nd, F.u, F.ub, F.ug, neu, F.bfl, F.n_bf);
  if (which == FL_PRES) return fl_grad(c, 1, F.p, F.pb, F.pg, neu, F.bfl, F.n_bf);
  return fl_grad(c, 1, F.q, F.qb, F.qg, neu, F.bfl, F.n_bf);
}

static int ff_zero(FlFlow &F) {
  FlCtx &c = *F.c;
  k_fl_fill<<<1024, BS, 0, c.stream>>>((size_t)c.nd * c.n, F.rhs, 0.0);
  k_fl_fill<<<1024, BS, 0, c.stream>>>((size_t)c.nnz, F.val, 0.0);
  FVK_HIP(hipGetLastError());
  return 0;
}

static int ff_source(FlFlow &F) {
  FlCtx &c = *F.c;
  k_fl_source<<<grid_for(c.n), BS, 0, c.stream>>>(c.n, c.nd, F.pg, c.vol, F.rhs);
  FVK_HIP(hipGetLastError());
  return 0;
}

static int ff_construct_pde(FlFlow &F) {
  FlCtx &c = *F.c;
  k_fl_pde_face<<<grid_for(c.nf), BS, 0, c.stream>>>(fl_geo(c), F.cfg.bl_c, F.u, F.ub, F.ug, F.spd, F.cc, F.ccb, F.cd,
                                                      F.cdb, F.val, F.fa, F.fb, F.fd, F.fcc, F.fdc);
  k_fl_pde_cell<<<grid_for(c.n), BS, 0, c.stream>>>(c.n, c.nf, c.nd, c.cptr, c.cfl, c.j1, c.jn, c.kii, F.fa, F.fb,
                                                     F.fd, F.fcc, F.fdc, F.u, F.cfg.urf_u, F.val, F.rhs, F.diag);
  FVK_HIP(hipGetLastError());
  return 0;
}

// FVK_ERR_HIP when a one-launch factorisation or sweep exceeded its wait
// bound (its results are then invalid)
static int fl_sweep_status(FlCtx &c) {
  int e = 0;
  IoCall call(c.io);
  int rc = c.io.get_raw(c.sweep_int + 3, sizeof e, &e);
  if (!rc) rc = c.io.finish();
  if (rc) return rc;
  if (e) {
    set_error("triangular sweep: a wait exceeded its bound; the preconditioner's results are invalid");
    return FVK_ERR_HIP;
  }
  return 0;
}

static int ff_solve(FlFlow &F, int isol, int ncmp, double *phi, double *rhs, int n_iter, double reduc, double *res0) {
  FlCtx &c = *F.c;
  int rc = fl_solve(c, isol, ncmp, F.val, phi, rhs, n_iter, reduc);
  if (rc) return rc;
  FlKS k[3];
  int failed = 0;
  IoCall call(c.io);
  if ((rc = c.io.get_raw(c.ks, sizeof(FlKS) * ncmp, k)) ||
      (rc = c.io.get_raw(c.sweep_int + 3, sizeof failed, &failed)) || (rc = c.io.finish()))
    return rc;
  for (int q = 0; q < ncmp; ++q) res0[q] = k[q].norm;
  return failed ? fl_sweep_status(c) : 0;
}

static int ff_construct_pp(FlFlow &F) {
  FlCtx &c = *F.c;
  k_fl_pp_face<<<grid_for(c.nf), BS, 0, c.stream>>>(fl_geo(c), F.u, F.ub, F.ug, F.p, F.pg, F.cc, F.ccb, F.diag,
                                                     F.spd, F.val, F.fa, F.fd, F.fdc);
  const int P = std::max(1, std::min(RG, (F.n_bf + RB - 1) / RB));
  k_fl_inout<<<P, RB, 0, c.stream>>>(F.n_bf, F.bfl, c.jn, c.btag, F.ccb, c.area, F.spd, c.part);
  k_fl_crat<<<1, RB, 0, c.stream>>>(P, c.part, c.scal);
  if (F.n_bf) k_fl_outlet<<<grid_for(F.n_bf), BS, 0, c.stream>>>(F.n_bf, F.bfl, c.jn, c.btag, c.scal, F.spd);
  k_fl_pp_cell<<<grid_for(c.n), BS, 0, c.stream>>>(c.n, c.nb, c.cptr, c.cfl, c.j1, c.jn, c.kii, c.btag, F.ccb, c.area,
                                                    F.spd, F.fa, F.fd, F.fdc, F.val, F.rhs);
  FVK_HIP(hipGetLastError());
  return 0;
}

static int ff_correct(FlFlow &F) {
  FlCtx &c = *F.c;
  k_fl_correct<<<grid_for(c.n), BS, 0, c.stream>>>(c.n, c.nd, F.qg, c.vol, F.diag, F.q, 0.0, F.cfg.urf_p, F.u, F.p);
  FVK_HIP(hipGetLastError());
  return 0;
}

// one outer iteration; res0[0..3]: the momentum and pressure-correction norms
static int ff_outer(FlFlow &F, double *res0) {
  FlCtx &c = *F.c;
  int rc;
  if ((rc = ff_zero(F))) return rc;
  if ((rc = ff_gradient(F, FL_PRES, 1))) return rc;
  if ((rc = ff_gradient(F, FL_VEL, 0))) return rc;
  if ((rc = ff_source(F))) return rc;
  if ((rc = ff_construct_pde(F))) return rc;
  if ((rc = ff_solve(F, 2, c.nd, F.u, F.rhs, F.cfg.n_iter_u, F.cfg.reduc_u, res0))) return rc;
  if ((rc = ff_zero(F))) return rc;
  if ((rc = ff_construct_pp(F))) return rc;
  k_fl_fill<<<1024, BS, 0, c.stream>>>((size_t)c.n, F.q, 0.0);
  if ((rc = ff_solve(F, 1, 1, F.q, F.rhs, F.cfg.n_iter_p, F.cfg.reduc_p, res0 + 3))) return rc;
  if ((rc = ff_gradient(F, FL_PP, 1))) return rc;
  if ((rc = ff_correct(F))) return rc;
  for (int k = 0; k < 4; ++k) F.res0[k] = res0[k];
  return 0;
}

}  // namespace fvk

// ---------------------------------------------------------------- C ABI
struct fvk_fl_mesh {
  fvk::FlMesh m;
};
struct fvk_fl_ctx {
  fvk::FlCtx c;
};
struct fvk_fl_flow {
  fvk::FlFlow f;
};

using namespace fvk;

extern "C" {

int fvk_fl_mesh_read_gmsh(const char *path, int n_dim, double l_sc, fvk_fl_mesh **out) {
  if (!path || !out) { set_error("null argument"); return FVK_ERR_ARG; }
  GmshRaw g;
  std::string e = parse_gmsh(g, path);
  if (!e.empty()) { set_error(e); return FVK_ERR_IO; }
  fvk_fl_mesh *m = new fvk_fl_mesh;
  e = fl_mesh_from_gmsh(m->m, g, n_dim, l_sc);
  if (!e.empty()) { delete m; set_error(e); return FVK_ERR_ARG; }
  *out = m;
  return FVK_OK;
}

int fvk_fl_mesh_from_records(int n_dim, int n_node, const double *x3, int n_elm, const int *e_ty, const int *e_tag,
                             const int *e_vptr, const int *e_vrt, fvk_fl_mesh **out) {
  if (!x3 || !e_ty || !e_tag || !e_vptr || !e_vrt || !out || n_node < 1 || n_elm < 1) {
    set_error("bad argument");
    return FVK_ERR_ARG;
  }
  static const int kNvrt[8] = {0, 2, 3, 4, 4, 8, 6, 5};
  GmshRaw g;
  g.node_id.resize(n_node);
  for (int i = 0; i < n_node; ++i) g.node_id[i] = i + 1;
  g.node_x.assign(x3, x3 + 3 * (size_t)n_node);
  g.e_vptr.assign(1, 0);
  for (int e = 0; e < n_elm; ++e) {
    if (e_ty[e] < 1 || e_ty[e] > 7 || e_vptr[e + 1] - e_vptr[e] != kNvrt[e_ty[e]]) {
      set_error("element " + std::to_string(e + 1) + ": bad type or vertex count");
      return FVK_ERR_ARG;
    }
    g.e_idx.push_back(e + 1);
    g.e_ty.push_back(e_ty[e]);
    g.e_tag0.push_back(e_tag[e]);
    for (int k = e_vptr[e]; k < e_vptr[e + 1]; ++k) g.e_vrt.push_back(e_vrt[k]);
    g.e_vptr.push_back((int)g.e_vrt.size());
  }
  fvk_fl_mesh *m = new fvk_fl_mesh;
  const std::string e = fl_mesh_from_gmsh(m->m, g, n_dim, 1.0);
  if (!e.empty()) { delete m; set_error(e); return FVK_ERR_ARG; }
  *out = m;
  return FVK_OK;
}

int fvk_fl_mesh_get_info(const fvk_fl_mesh *mm, int *info) {
  if (!mm || !info) { set_error("null argument"); return FVK_ERR_ARG; }
  const FlMesh &m = mm->m;
  info[0] = m.n_dim; info[1] = m.n_vrt; info[2] = m.n_bnd; info[3] = m.n_dmn; info[4] = m.n_fce;
  info[5] = (int)m.ng_col.size(); info[6] = (int)m.elm_vrt.size(); info[7] = (int)m.fce_vrt.size();
  return FVK_OK;
}

int fvk_fl_mesh_get_arrays(const fvk_fl_mesh *mm, double *x3, int *elm_vptr, int *elm_vrt, int *bnd_tag,
                           int *fce_elm, int *fce_vptr, int *fce_vrt, int *ng_ptr, int *ng_col, int *elm_idx) {
  if (!mm) { set_error("null argument"); return FVK_ERR_ARG; }
  const FlMesh &m = mm->m;
  auto cp = [](const auto &v, auto *dst) { if (dst) std::copy(v.begin(), v.end(), dst); };
  cp(m.x, x3); cp(m.elm_vptr, elm_vptr); cp(m.elm_vrt, elm_vrt); cp(m.bnd_tag, bnd_tag); cp(m.fce_elm, fce_elm);
  cp(m.fce_vptr, fce_vptr); cp(m.fce_vrt, fce_vrt); cp(m.ng_ptr, ng_ptr); cp(m.ng_col, ng_col);
  cp(m.elm_idx, elm_idx);
  return FVK_OK;
}

void fvk_fl_mesh_free(fvk_fl_mesh *m) { delete m; }

int fvk_fl_ctx_create(int n_dim, int n_vrt, const double *x3, int n_bnd, const int *bnd_tag, int n_dmn,
                      const int *elm_vptr, const int *elm_vrt, int n_fce, const int *fce_elm, const int *fce_vptr,
                      const int *fce_vrt, const int *ng_ptr, const int *ng_col, int device, fvk_fl_ctx **out) {
  if (!x3 || !elm_vptr || !elm_vrt || !fce_elm || !fce_vptr || !fce_vrt || !ng_ptr || !ng_col || !out ||
      (n_bnd > 0 && !bnd_tag) || (n_dim != 2 && n_dim != 3) || n_dmn < 1 || n_fce < 1 || n_vrt < 1 || n_bnd < 0) {
    set_error("bad argument");
    return FVK_ERR_ARG;
  }
  fvk_fl_ctx *cc = new fvk_fl_ctx;
  FlCtx &c = cc->c;
  c.device = device;
  hipError_t e = hipSetDevice(device);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&c.stream, hipStreamNonBlocking);
  if (e != hipSuccess) { delete cc; set_error(hipGetErrorString(e)); return FVK_ERR_HIP; }
  c.io.stream = c.stream;
  const int rc = fl_ctx_build(c, n_dim, n_vrt, x3, n_bnd, bnd_tag, n_dmn, elm_vptr, elm_vrt, n_fce, fce_elm, fce_vptr,
                              fce_vrt, ng_ptr, ng_col);
  if (rc) { fl_ctx_free(c); delete cc; return rc; }
  *out = cc;
  return FVK_OK;
}

int fvk_fl_csr_create(int n, const int *ia, const int *ja, int device, fvk_fl_ctx **out) {
  if (!ia || !ja || !out || n < 1) { set_error("bad argument"); return FVK_ERR_ARG; }
  fvk_fl_ctx *cc = new fvk_fl_ctx;
  FlCtx &c = cc->c;
  c.device = device;
  hipError_t e = hipSetDevice(device);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&c.stream, hipStreamNonBlocking);
  if (e != hipSuccess) { delete cc; set_error(hipGetErrorString(e)); return FVK_ERR_HIP; }
  c.io.stream = c.stream;
  const int rc = fl_csr_setup(c, n, ia, ja);
  if (rc) { fl_ctx_free(c); delete cc; return rc; }
  *out = cc;
  return FVK_OK;
}

int fvk_sweep_plan(int n, const int *ia, const int *ja, int max_rows, int *info) {
  if (!ia || !ja || !info || n < 1 || max_rows < 64) { set_error("bad argument"); return FVK_ERR_ARG; }
  FlPattern q;
  const int rc = fl_pattern(n, ia, ja, q);
  if (rc) return rc;
  const SweepGraph g = fl_sweep_graph(n, q.ia, q.ja, q.klo, q.kup, q.tpos);
  SweepPlan p;
  std::string e = sweep_plan(g, max_rows, p);
  if (!e.empty()) { set_error(e); return FVK_ERR_ARG; }
  e = sweep_plan_check(g, p);
  if (!e.empty()) { set_error("sweep plan: " + e); return FVK_ERR_STATE; }
  const int v[8] = {p.P, p.np / p.width, p.levels, p.bricks ? 1 : 0, (int)p.lds(1), (int)p.lds(3), p.d[0].NE, p.d[1].NE};
  std::copy(v, v + 8, info);
  return FVK_OK;
}

int fvk_sweep_positions(int n, const int *ia, const int *ja, int max_rows, int64_t limit, int64_t *positions) {
  if (!ia || !ja || !positions || n < 1 || max_rows < 64 || limit < 0) { set_error("bad argument"); return FVK_ERR_ARG; }
  FlPattern q;
  const int rc = fl_pattern(n, ia, ja, q);
  if (rc) return rc;
  SweepPlan p;
  const std::string e = sweep_plan(fl_sweep_graph(n, q.ia, q.ja, q.klo, q.kup, q.tpos), max_rows, p, (long)limit);
  if (!e.empty()) { set_error(e); return FVK_ERR_ARG; }
  *positions = p.np;
  return FVK_OK;
}

int fvk_sweep_times(int n, const int *ia, const int *ja, int max_rows, double *us) {
  if (!ia || !ja || !us || n < 1 || max_rows < 64) { set_error("bad argument"); return FVK_ERR_ARG; }
  FlPattern q;
  const int rc = fl_pattern(n, ia, ja, q);
  if (rc) return rc;
  SweepPlan p;
  const std::string e = sweep_plan(fl_sweep_graph(n, q.ia, q.ja, q.klo, q.kup, q.tpos), max_rows, p);
  if (!e.empty()) { set_error(e); return FVK_ERR_ARG; }
  us[0] = sweep_plan_us(p);
  us[1] = p.chunk_us;
  return FVK_OK;
}

int fvk_fl_csr_matches(const fvk_fl_ctx *cc, int n, const int *ia, const int *ja) {
  if (!cc || !ia || !ja) return 0;
  const FlCtx &c = cc->c;
  if (n != c.n || ia[n] - 1 != c.nnz) return 0;
  for (int i = 0; i <= n; ++i)
    if (ia[i] - 1 != c.h_ia[i]) return 0;
  for (int k = 0; k < c.nnz; ++k)
    if (ja[k] - 1 != c.h_ja[k]) return 0;
  return 1;
}

void fvk_fl_ctx_destroy(fvk_fl_ctx *cc) {
  if (!cc) return;
  fl_ctx_free(cc->c);
  delete cc;
}

int fvk_fl_geometry(fvk_fl_ctx *cc, double *x_vc, double *vol, double *x_fc, double *norm, double *area, double *x_pc,
                    double *x_nc, double *l_pn, double *w_fp, double *ls) {
  if (!cc) { set_error("null argument"); return FVK_ERR_ARG; }
  FlCtx &c = cc->c;
  const int nd = c.nd;
  int rc = 0;
  IoCall call(c.io);
  if (x_vc && (rc = fl_out(c, c.xvc, nd, c.n, x_vc))) return rc;
  if (vol && (rc = fl_out(c, c.vol, 1, c.n, vol))) return rc;
  if (x_fc && (rc = fl_out(c, c.xfc, nd, c.nf, x_fc))) return rc;
  if (norm && (rc = fl_out(c, c.nrm, nd, c.nf, norm))) return rc;
  if (area && (rc = fl_out(c, c.area, 1, c.nf, area))) return rc;
  if (x_pc && (rc = fl_out(c, c.xpc, nd, c.nf, x_pc))) return rc;
  if (x_nc && (rc = fl_out(c, c.xnc, nd, c.nf, x_nc))) return rc;
  if (l_pn && (rc = fl_out(c, c.lpn, 1, c.nf, l_pn))) return rc;
  if (w_fp && (rc = fl_out(c, c.wfp, 1, c.nf, w_fp))) return rc;
  if (ls && (rc = fl_out(c, c.ls, nd * nd, c.n, ls))) return rc;
  return c.io.finish();
}

int fvk_fl_ls_gradient(fvk_fl_ctx *cc, int n_cmp, const double *phi, double *phi_bnd, double *grad, int neu_bnd) {
  if (!cc || !phi || !grad || (!phi_bnd && cc->c.nb > 0) || n_cmp < 1 || n_cmp > 3) {
    set_error("bad argument");
    return FVK_ERR_ARG;
  }
  FlCtx &c = cc->c;
  double *d = wkv(c, 0), *dg = wkv(c, 2);
  int rc = 0;
  if (!c.bval) {
    std::vector<int> bfl;
    for (int f = 0; f < c.nf; ++f)
      if (c.h_jn[f] < 0) bfl.push_back(f);
    c.n_bf = (int)bfl.size();
    if ((rc = fl_up(c, &c.bfl, bfl))) return rc;
    if ((rc = fl_alloc(c, &c.bval, (size_t)3 * std::max(c.nb, 1)))) return rc;
  }
  IoCall call(c.io);
  if ((rc = fl_in(c, phi, n_cmp, c.n, d))) return rc;
  if (c.nb && (rc = fl_in(c, phi_bnd, n_cmp, c.nb, c.bval))) return rc;
  if ((rc = fl_grad(c, n_cmp, d, c.bval, dg, neu_bnd, c.bfl, c.n_bf))) return rc;
  if ((rc = fl_out(c, dg, c.nd * n_cmp, c.n, grad))) return rc;
  if (neu_bnd && c.nb && (rc = fl_out(c, c.bval, n_cmp, c.nb, phi_bnd))) return rc;
  return c.io.finish();
}

int fvk_fl_lin_eqns_solver(fvk_fl_ctx *cc, const double *a_ij, double *phi, double *rhs, double *norm, int n_iter,
                           double reduc, int isol) {
  if (!cc || !a_ij || !phi || !rhs || !norm || n_iter < 0 || (isol != 1 && isol != 2)) {
    set_error("bad argument");
    return FVK_ERR_ARG;
  }
  FlCtx &c = cc->c;
  int rc = 0;
  if (!c.lin && (rc = fl_alloc(c, &c.lin, (size_t)c.nnz + 2 * (size_t)c.n))) return rc;
  double *da = c.lin, *dphi = da + c.nnz, *drhs = dphi + c.n;
  IoCall call(c.io);
  if ((rc = fl_in(c, a_ij, 1, c.nnz, da)) || (rc = fl_in(c, phi, 1, c.n, dphi)) || (rc = fl_in(c, rhs, 1, c.n, drhs)))
    return rc;
  if ((rc = fl_solve(c, isol, 1, da, dphi, drhs, n_iter, reduc))) return rc;
  FlKS k;
  int failed = 0;
  if ((rc = fl_out(c, dphi, 1, c.n, phi)) || (rc = fl_out(c, drhs, 1, c.n, rhs))) return rc;
  if ((rc = c.io.get_raw(c.ks, sizeof k, &k)) || (rc = c.io.get_raw(c.sweep_int + 3, sizeof failed, &failed))) return rc;
  if ((rc = c.io.finish())) return rc;
  *norm = k.norm;
  return failed ? fl_sweep_status(c) : FVK_OK;
}

int fvk_fl_ctx_set_param(fvk_fl_ctx *cc, const char *name, double value) {
  if (!cc || !name) { set_error("null argument"); return FVK_ERR_ARG; }
  FlCtx &c = cc->c;
  if (!std::strcmp(name, "sweep_one_launch") && (value == 0 || value == 1)) {
    if (value == 1) {
      int mx = 0;
      for (int i = 0; i < c.n; ++i) {
        int lo = c.h_ia[i], up = c.h_ia[i + 1];
        while (lo < c.h_ia[i + 1] && c.h_ja[lo] < i) ++lo;
        while (up > c.h_ia[i] && c.h_ja[up - 1] > i) --up;
        mx = std::max({mx, lo - c.h_ia[i], c.h_ia[i + 1] - up});
      }
      if (mx > kSweepSlots) { set_error("a row has more lower or upper entries than one launch holds"); return FVK_ERR_ARG; }
    }
    c.one_launch = value != 0;
    return FVK_OK;
  }
  if (!std::strcmp(name, "sweep_parts") && (value == 0 || value == 1 || value == 2)) {
    if (value != 0 && !c.narrow) { set_error("a row has more lower or upper entries than one launch holds"); return FVK_ERR_ARG; }
    const bool plan = (value == 2) != (c.parts == 2);
    c.parts = (int)value;
    if (!plan) return FVK_OK;
    FVK_HIP(hipStreamSynchronize(c.stream));
    return fl_parts_setup(c);
  }
  if (!std::strcmp(name, "sweep_part_rows") && value >= 256 && value <= 6400 && value == (int)value) {
    if (!c.narrow) { set_error("a row has more lower or upper entries than one launch holds"); return FVK_ERR_ARG; }
    FVK_HIP(hipStreamSynchronize(c.stream));
    c.part_rows = (int)value;
    return fl_parts_setup(c);
  }
  if (!std::strcmp(name, "sweep_positions") && value >= 0 && value <= 1 << 28 && value == (long)value) {
    if (!c.narrow) { set_error("a row has more lower or upper entries than one launch holds"); return FVK_ERR_ARG; }
    FVK_HIP(hipStreamSynchronize(c.stream));
    c.positions = (long)value;
    return fl_parts_setup(c);
  }
  if (!std::strcmp(name, "sweep_blocks") && value >= 0 && value <= 65536 && value == (int)value) {
    c.sweep_blocks = c.sw.blocks = (int)value;
    return FVK_OK;
  }
  if (!std::strcmp(name, "sweep_fail") && value == 2) {
    c.sw.deny = true;
    return FVK_OK;
  }
  if (!std::strcmp(name, "sweep_fail") && value == 1 && c.sweep_int) {
    const int one = 1;
    FVK_HIP(hipMemcpyAsync(c.sweep_int + 3, &one, sizeof one, hipMemcpyHostToDevice, c.stream));
    FVK_HIP(hipStreamSynchronize(c.stream));
    return FVK_OK;
  }
  set_error(std::string("unknown parameter or value out of range: ") + name);
  return FVK_ERR_ARG;
}

int fvk_fl_flow_create(fvk_fl_ctx *cc, const double *params, fvk_fl_flow **out) {
  if (!cc || !params || !out) { set_error("null argument"); return FVK_ERR_ARG; }
  FlCfg cfg;
  cfg.cc = params[0]; cfg.cd = params[1]; cfg.urf_u = params[2]; cfg.urf_p = params[3]; cfg.bl_c = params[4];
  cfg.n_iter_u = (int)params[5]; cfg.reduc_u = params[6]; cfg.n_iter_p = (int)params[7]; cfg.reduc_p = params[8];
  if (!(cfg.urf_u > 0.0) || cfg.n_iter_u < 0 || cfg.n_iter_p < 0) { set_error("bad flow parameters"); return FVK_ERR_ARG; }
  fvk_fl_flow *ff = new fvk_fl_flow;
  ff->f.c = &cc->c;
  ff->f.cfg = cfg;
  const int rc = ff_build(ff->f);
  if (rc) { ff_free(ff->f); delete ff; return rc; }
  *out = ff;
  return FVK_OK;
}

void fvk_fl_flow_destroy(fvk_fl_flow *ff) {
  if (!ff) return;
  ff_free(ff->f);
  delete ff;
}

int fvk_fl_flow_set(fvk_fl_flow *ff, const double *vel, const double *vel_bnd, const double *pres,
                    const double *pres_bnd) {
  if (!ff) { set_error("null argument"); return FVK_ERR_ARG; }
  FlFlow &F = ff->f;
  FlCtx &c = *F.c;
  int rc = 0;
  if (vel && (rc = fl_in(c, vel, c.nd, c.n, F.u))) return rc;
  if (vel_bnd && c.nb && (rc = fl_in(c, vel_bnd, c.nd, c.nb, F.ub))) return rc;
  if (pres && (rc = fl_in(c, pres, 1, c.n, F.p))) return rc;
  if (pres_bnd && c.nb && (rc = fl_in(c, pres_bnd, 1, c.nb, F.pb))) return rc;
  return FVK_OK;
}

int fvk_fl_flow_get(fvk_fl_flow *ff, double *vel, double *vel_bnd, double *pres, double *pres_bnd, double *pp,
                    double *spd) {
  if (!ff) { set_error("null argument"); return FVK_ERR_ARG; }
  FlFlow &F = ff->f;
  FlCtx &c = *F.c;
  int rc = 0;
  IoCall call(c.io);
  if (vel && (rc = fl_out(c, F.u, c.nd, c.n, vel))) return rc;
  if (vel_bnd && c.nb && (rc = fl_out(c, F.ub, c.nd, c.nb, vel_bnd))) return rc;
  if (pres && (rc = fl_out(c, F.p, 1, c.n, pres))) return rc;
  if (pres_bnd && c.nb && (rc = fl_out(c, F.pb, 1, c.nb, pres_bnd))) return rc;
  if (pp && (rc = fl_out(c, F.q, 1, c.n, pp))) return rc;
  if (spd && (rc = fl_out(c, F.spd, 1, c.nf, spd))) return rc;
  return c.io.finish();
}

// intermediate arrays of the current iteration: the matrix values (nnz),
// the right-hand side (n_dim x n_dmn), 1/a_P (n_dmn), the gradients of
// velocity, pressure and pressure correction
int fvk_fl_flow_get_system(fvk_fl_flow *ff, double *val, double *rhs, double *diag, double *vel_grad,
                           double *pres_grad, double *pp_grad, double *pp_bnd) {
  if (!ff) { set_error("null argument"); return FVK_ERR_ARG; }
  FlFlow &F = ff->f;
  FlCtx &c = *F.c;
  int rc = 0;
  IoCall call(c.io);
  if (val && (rc = fl_out(c, F.val, 1, c.nnz, val))) return rc;
  if (rhs && (rc = fl_out(c, F.rhs, c.nd, c.n, rhs))) return rc;
  if (diag && (rc = fl_out(c, F.diag, 1, c.n, diag))) return rc;
  if (vel_grad && (rc = fl_out(c, F.ug, c.nd * c.nd, c.n, vel_grad))) return rc;
  if (pres_grad && (rc = fl_out(c, F.pg, c.nd, c.n, pres_grad))) return rc;
  if (pp_grad && (rc = fl_out(c, F.qg, c.nd, c.n, pp_grad))) return rc;
  if (pp_bnd && c.nb && (rc = fl_out(c, F.qb, 1, c.nb, pp_bnd))) return rc;
  return c.io.finish();
}

// One step of navierstokes' outer loop, by name of the reference routine
// it replaces: 0 zero (rhs and matrix), 1 ls_gradient(pres, neu 1),
// 2 ls_gradient(vel, neu 0), 3 ns_source, 4 construct_pde, 5 momentum
// solves (res0[0..n_dim)), 6 construct_pp, 7 pressure-correction solve
// (res0[0]), 8 ls_gradient(pp, neu 1), 9 ns_correction
int fvk_fl_flow_step(fvk_fl_flow *ff, int step, double *res0) {
  if (!ff || step < 0 || step > 9 || ((step == 5 || step == 7) && !res0)) { set_error("bad argument"); return FVK_ERR_ARG; }
  FlFlow &F = ff->f;
  FlCtx &c = *F.c;
  int rc = 0;
  switch (step) {
    case 0: rc = ff_zero(F); break;
    case 1: rc = ff_gradient(F, FL_PRES, 1); break;
    case 2: rc = ff_gradient(F, FL_VEL, 0); break;
    case 3: rc = ff_source(F); break;
    case 4: rc = ff_construct_pde(F); break;
    case 5: rc = ff_solve(F, 2, c.nd, F.u, F.rhs, F.cfg.n_iter_u, F.cfg.reduc_u, res0); break;
    case 6: rc = ff_construct_pp(F); break;
    case 7:
      k_fl_fill<<<1024, BS, 0, c.stream>>>((size_t)c.n, F.q, 0.0);
      rc = ff_solve(F, 1, 1, F.q, F.rhs, F.cfg.n_iter_p, F.cfg.reduc_p, res0);
      break;
    case 8: rc = ff_gradient(F, FL_PP, 1); break;
    case 9: rc = ff_correct(F); break;
  }
  if (!rc) FVK_HIP(hipStreamSynchronize(c.stream));
  return rc;
}

// n outer iterations of navierstokes.f90:515-641 with fp_iter_ctrl's exit
// rule (:806-845) for n_iter and res_drop; res0: 4 norms per iteration,
// norm_gl: the normalised residual per iteration; *n_done: iterations run
int fvk_fl_flow_run(fvk_fl_flow *ff, int n_iter, double res_drop, double *res0, double *norm_gl, int *n_done) {
  if (!ff || n_iter < 1 || !n_done) { set_error("bad argument"); return FVK_ERR_ARG; }
  FlFlow &F = ff->f;
  double norm_mx = 0.0;
  int fp_exit = 0, it;
  for (it = 1; it <= n_iter; ++it) {
    double r[4];
    int rc = ff_outer(F, r);
    if (rc) return rc;
    if (res0)
      for (int k = 0; k < 4; ++k) res0[4 * (it - 1) + k] = r[k];
    double gl = r[0];
    for (int k = 1; k < 4; ++k) gl = std::max(gl, r[k]);
    gl = std::max(gl, 0.0);  // res0(5:10) are zero
    norm_mx = std::max(norm_mx, gl);
    gl = gl / (norm_mx + SMALL);
    if (norm_gl) norm_gl[it - 1] = gl;
    if (gl < res_drop || it > n_iter - 2) ++fp_exit;
    if (fp_exit > 1) break;
  }
  *n_done = std::min(it, n_iter);
  return FVK_OK;
}

}  // extern "C"
