"""The FP64 Krylov kernels around the sizes where their launch changes: a
block that is not full, one row more than a block of 256, a grid rounded up to
a multiple of 8 (its last blocks without rows), and both sides of the changes
to blocks of 512 (1024 * 256 rows) and of 1024 (1024 * 512 rows)."""
import numpy as np
import pytest

from tests.helpers import require_lib
from tests.test_gpu_sweeps import random_matrix

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def mult(m, pl, gp, gn):
    t = m.topology()
    inner = t["fce_in"] > 0
    a, b, gp, gn = t["fce_ip"][inner] - 1, t["fce_in"][inner] - 1, gp[inner], gn[inner]
    n = m.n_vol
    return lambda x: pl * x + np.bincount(a, gp * x[b], n) + np.bincount(b, gn * x[a], n)


def pcg(A, c, b, steps):
    x, r = np.zeros_like(b), b.copy()
    z = c * r
    p, s = z.copy(), r @ z
    for _ in range(steps):
        q = A(p)
        al = s / (p @ q)
        x += al * p
        r -= al * q
        z = c * r
        s, so = r @ z, s
        p = z + s / so * p
    return x


@pytest.mark.parametrize("dims", [(3, 1, 1), (257, 1, 1), (4097, 1, 1), (64, 64, 64), (4097, 8, 8), (64, 64, 128), (4097, 8, 16)])
def test_two_steps(dims):
    fvk = require_lib()
    print("krylov sizes:", dims, flush=True)
    m = fvk.Mesh.box(*dims, jitter=0.0, seed=1)
    n = m.n_vol
    ctx = fvk.grd_solv(m)
    pl, gp, gn = random_matrix(m, 5)
    b = np.random.default_rng(n).standard_normal((n, 3))
    # a rounding error per addition of a reduction, four reductions; the
    # rows' own errors are below 1e-14
    tol = 4 * n * EPS + 1e-14

    pls = pl + 6.0  # dominant for the symmetric matrix too
    fvk.set_matrix(ctx, pls, gp, gp)
    A = mult(m, pls, gp, gp)
    for k in (1, 2, 3):
        x, r = np.zeros((n, k)), b[:, :k].copy()
        fvk.solv_cg(ctx, 0, 1e-30, 2, x, r)
        assert np.array_equal(r, b[:, :k])  # from x = 0 the initial residual is b
        for q in range(k):
            want = pcg(A, 1.0 / pls, b[:, q], 2)
            assert np.abs(x[:, q] - want).max() <= tol * np.abs(want).max(), (k, q)

    fvk.set_matrix(ctx, pl, gp, gn)
    A = mult(m, pl, gp, gn)
    x, r = np.zeros((n, 3)), b.copy()
    fvk.solv_bicg(ctx, 0, 1e-30, 1, x, r)
    for q in range(3):
        # one step: p = r = b, gamma = r.r0 / u.r0, omega = v.s / v.v
        b0, c = b[:, q], 1.0 / pl
        u = A(c * b0)
        g = b0 @ b0 / (u @ b0)
        s = b0 - g * u
        v = A(c * s)
        want = g * c * b0 + (v @ s) / (v @ v) * c * s
        assert np.abs(x[:, q] - want).max() <= tol * np.abs(want).max(), q
    ctx.destroy()


@pytest.mark.parametrize("imat", [0, 1])
@pytest.mark.parametrize("fn,n_iter", [("solv_cg", 30), ("solv_bicg", 12)])
def test_stops_as_if_told_the_iterations(fn, n_iter, imat):
    """A solve that meets its tolerance after k iterations leaves the bits of
    a solve of exactly k iterations, for an end at the start, in the middle
    and at the last iteration allowed (the host sees the end while later
    iterations are queued)."""
    fvk = require_lib()
    m = fvk.Mesh.box(20, 17, 13, jitter=0.05, seed=2)
    ctx = fvk.grd_solv(m)
    pl, gp, gn = random_matrix(m, 9)
    sym = fn == "solv_cg"
    fvk.set_matrix(ctx, pl + 6.0 * sym, gp, gp if sym else gn)
    b = np.random.default_rng(1).standard_normal((m.n_vol, 2))
    pc = imat if sym else 2 * imat

    def run(reduc, its):
        x, r = np.zeros((m.n_vol, 2)), b.copy()
        rn, st = getattr(fvk, fn)(ctx, pc, reduc, its, x, r)
        return x, r, list(st.iters[:2])

    seen = set()
    for reduc in (2.0, 0.3, 1e-2, 1e-4, 1e-30):
        x, r, k = run(reduc, n_iter)
        seen.update(k)
        for q in range(2):
            xk, rk, kk = run(0.0, k[q])
            assert kk[q] == k[q] and np.array_equal(xk[:, q], x[:, q]) and np.array_equal(rk[:, q], r[:, q])
    assert 1 in seen and n_iter in seen and len(seen) > 3
    ctx.destroy()
