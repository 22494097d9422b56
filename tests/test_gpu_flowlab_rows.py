"""flowlab's CG and BiCGStab on patterns of every row width the matrix product
is laid out for: the most entries of a row at and around 4, 5, 7 and 8 (by
slots), 9 (CSR), and a pattern that is mostly empty slots (CSR), with one
row, fewer rows than a block has threads, and several blocks; solves that stop
on the norm and solves that run all their iterations.  Against the same
recurrences in numpy."""
import ctypes as C

import numpy as np
import pytest

from tests.helpers import require_lib

pytestmark = pytest.mark.gpu
SMALL = float.fromhex("0x1.79ca10c924224p-67")
EPS = np.finfo(float).eps


def pattern(n, width, full, seed):
    """1-based CSR with sorted columns, symmetric, with a diagonal: at most
    `width` entries a row; full: most rows near that width, else few."""
    rng = np.random.default_rng(seed)
    cols = [{i} for i in range(n)]
    for i in range(n):
        for j in i + 1 + rng.permutation(min(40, n - 1 - i) if i < n - 1 else 0):
            if (full or i % 50 == 0) and len(cols[i]) < width and len(cols[j]) < width:
                cols[i].add(int(j))
                cols[j].add(i)
    ia, ja = [1], []
    for c in cols:
        ja += [j + 1 for j in sorted(c)]
        ia.append(len(ja) + 1)
    return np.array(ia, np.int32), np.array(ja, np.int32)


class Ref:
    def __init__(self, ia, ja, a):
        self.n = n = len(ia) - 1
        self.rows = [[(int(ja[k]) - 1, a[k]) for k in range(ia[i] - 1, ia[i + 1] - 1)] for i in range(n)]
        self.at = [dict(r) for r in self.rows]
        self.r = np.repeat(np.arange(n), np.diff(ia))
        self.c, self.a = ja - 1, a
        self.pc = np.zeros(n)
        for i in range(n):
            s = self.at[i][i]
            for j, v in self.rows[i]:
                if j < i:
                    s -= v * self.pc[j] * self.at[j][i]
            self.pc[i] = 1.0 / (s + SMALL)

    def mv(self, x):
        return np.bincount(self.r, self.a * x[self.c], self.n)

    def direct(self, b):
        x, y = np.zeros(self.n), np.zeros(self.n)
        for i in range(self.n):
            x[i] = (b[i] - sum(v * x[j] for j, v in self.rows[i] if j < i)) * self.pc[i]
        for i in range(self.n - 1, -1, -1):
            y[i] = (x[i] / (self.pc[i] + SMALL) - sum(v * y[j] for j, v in self.rows[i] if j > i)) * self.pc[i]
        return y

    def solve(self, x, b, n_iter, reduc, isol):
        x = x.copy()
        r0 = b - self.mv(x)
        r, norm0, its = r0.copy(), np.abs(r0).sum(), 0
        norm, p, u = norm0, np.zeros(self.n), np.zeros(self.n)
        s, al, be, ga = 1.0 / SMALL, 1.0, 1.0, 1.0
        for _ in range(n_iter):
            if isol == 1:
                z = self.direct(r)
                so, s = s, z @ r
                p = z + s / (so + SMALL) * p
                q = self.mv(p)
                a = s / (p @ q + SMALL)
                x, r = x + a * p, r - a * q
            else:
                bo, be = be, r @ r0
                p = r + be * ga / (al * bo + SMALL) * (p - al * u)
                z = self.direct(p)
                u = self.mv(z)
                ga = be / (u @ r0 + SMALL)
                x, r = x + ga * z, r - ga * u
                z = self.direct(r)
                v = self.mv(z)
                al = v @ r / (((v + SMALL) ** 2).sum() + SMALL)
                x, r = x + al * z, r - al * v
            norm, its = np.abs(r).sum(), its + 1
            if norm / (norm0 + SMALL) < reduc:
                break
        return x, r0, norm, its


@pytest.mark.parametrize("n,width,full", [(1, 1, True), (70, 4, True), (700, 5, True), (700, 6, True), (700, 7, True),
                                          (1100, 8, True), (600, 9, True), (600, 8, False)])
def test_solves_by_row_width(n, width, full):
    fvk = require_lib()
    print("flowlab rows:", n, width, full, flush=True)
    ia, ja = pattern(n, width, full, 7)
    rows = np.repeat(np.arange(n), np.diff(ia))
    rng = np.random.default_rng(n)
    a = rng.uniform(-1.0, -0.2, len(ja))
    low = np.minimum(rows, ja - 1) * n + np.maximum(rows, ja - 1)  # one value per pair for the symmetric matrix
    _, first = np.unique(low, return_inverse=True)
    sym = a[first]
    L = fvk.lib()
    h = C.c_void_p()
    ip = lambda v: v.ctypes.data_as(C.POINTER(C.c_int))
    dp = lambda v: v.ctypes.data_as(C.POINTER(C.c_double))
    assert L.fvk_fl_csr_create(n, ip(ia), ip(ja), 0, C.byref(h)) == 0
    for isol, vals in ((1, sym), (2, a)):
        vals = vals.copy()
        off = rows != ja - 1
        vals[~off] = 0.5 + np.bincount(rows[off], np.abs(vals[off]), n)
        ref = Ref(ia, ja, vals)
        b, x0 = rng.standard_normal(n), rng.standard_normal(n)
        for n_iter, reduc in ((0, 1e-3), (1, 0.0), (3, 0.0), (25, 1e-3)):
            x, r, norm = x0.copy(), b.copy(), np.zeros(1)
            assert L.fvk_fl_lin_eqns_solver(h, dp(vals), dp(x), dp(r), dp(norm), n_iter, C.c_double(reduc), isol) == 0
            wx, wr, wn, its = ref.solve(x0, b, n_iter, reduc, isol)
            # rounding of sums of n terms, passed on by up to `its` iterations
            # of a system whose condition number is below 100
            tol = 100 * max(its, 1) * n * EPS
            assert np.abs(r - wr).max() <= tol * np.abs(wr).max()
            assert np.abs(x - wx).max() <= tol * np.abs(wx).max(), (isol, n_iter)
            assert abs(norm[0] - wn) <= tol * np.abs(wr).sum(), (isol, n_iter)
    L.fvk_fl_ctx_destroy(h)


def scattered(nx):
    """The pattern of a box of nx^3 cells numbered at random."""
    k = np.random.default_rng(2).permutation(nx ** 3).reshape(nx, nx, nx)
    e = np.concatenate([np.stack([a.ravel(), b.ravel()], 1) for a, b in ((k[1:], k[:-1]), (k[:, 1:], k[:, :-1]),
                                                                        (k[:, :, 1:], k[:, :, :-1]))])
    r, c = np.concatenate([e[:, 0], e[:, 1], k.ravel()]), np.concatenate([e[:, 1], e[:, 0], k.ravel()])
    o = np.lexsort((c, r))
    return (1 + np.concatenate([[0], np.cumsum(np.bincount(r))])).astype(np.int32), (c[o] + 1).astype(np.int32)


@pytest.mark.parametrize("ia,ja", [pattern(900, 7, True, 3), scattered(16)])
def test_sweep_forms_bitwise(ia, ja):
    """One launch per level, chunks, parts, and a pattern with more positions
    than the parts' tables may hold ("sweep_positions") or tables that find no
    memory ("sweep_fail" 2), which take chunks."""
    fvk = require_lib()
    n = len(ia) - 1
    rows = np.repeat(np.arange(n), np.diff(ia))
    rng = np.random.default_rng(5)
    a, b = rng.uniform(-1.0, -0.2, len(ja)), rng.standard_normal(n)
    a[rows == ja - 1] = 9.0
    L = fvk.lib()
    h = C.c_void_p()
    ip = lambda v: v.ctypes.data_as(C.POINTER(C.c_int))
    dp = lambda v: v.ctypes.data_as(C.POINTER(C.c_double))
    assert L.fvk_fl_csr_create(n, ip(ia), ip(ja), 0, C.byref(h)) == 0
    first = None
    for params in ((), ((b"sweep_positions", 64),), ((b"sweep_positions", 0),), ((b"sweep_parts", 0),), ((b"sweep_parts", 2),),
                   ((b"sweep_positions", 64), (b"sweep_parts", 2)), ((b"sweep_fail", 2), (b"sweep_positions", 0)),
                   ((b"sweep_part_rows", 300),), ((b"sweep_one_launch", 0),)):
        print("flowlab sweeps:", params, flush=True)
        for k, v in params:
            assert L.fvk_fl_ctx_set_param(h, k, C.c_double(v)) == 0
        x, r, norm = np.zeros(n), b.copy(), np.zeros(1)
        assert L.fvk_fl_lin_eqns_solver(h, dp(a), dp(x), dp(r), dp(norm), 4, C.c_double(0.0), 2) == 0
        first = x if first is None else first
        assert np.array_equal(x, first), params
    L.fvk_fl_ctx_destroy(h)
