"""The plan of the one-launch triangular sweeps (host only): which rows a
block walks together and which values pass between blocks.  fvk_sweep_plan
walks every plan as the kernels do and fails when a value would be read
before it is there, when a part needs a part taken after it, or when a row
is not run once; the cases are where that can go wrong: one row, one part,
ragged boxes, chains, unstructured and unsorted patterns, rows with one to
eight entries on a side."""
import resource
import subprocess
import sys

import numpy as np
import pytest

from programs_amd import fvk
from tests.helpers import ROOT

LDS = 163840  # bytes of LDS of a compute unit


def csr(n, pairs, unsorted=None):
    """1-based CSR of the pattern pairs + transposed + diagonal; unsorted: a
    generator that shuffles the columns of some rows."""
    cols = [{i} for i in range(n)]
    for i, j in pairs:
        cols[i].add(j)
        cols[j].add(i)
    ia, ja = [1], []
    for c in cols:
        c = sorted(c)
        if unsorted is not None and unsorted.random() < 0.3:
            unsorted.shuffle(c)
        ja += [j + 1 for j in c]
        ia.append(len(ja) + 1)
    return ia, ja


def box(nx, ny, nz):
    k = np.arange(nx * ny * nz).reshape(nz, ny, nx)
    e = [(k[:, :, 1:], k[:, :, :-1]), (k[:, 1:], k[:, :-1]), (k[1:], k[:-1])]
    return nx * ny * nz, np.concatenate([np.stack([a.ravel(), b.ravel()], 1) for a, b in e])


@pytest.mark.parametrize("rows", [64, 100, 1728, 6400])
@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 1, 1), (65, 1, 1), (7, 5, 3), (13, 12, 11), (40, 33, 1), (25, 24, 23)])
def test_boxes(dims, rows):
    n, pairs = box(*dims)
    p = fvk.sweep_plan(*csr(n, pairs.tolist()), rows)
    assert p["levels"] == sum(dims) - 2
    assert p["lds3"] <= LDS and p["chunks"] * 64 >= n
    if min(dims) > 1:
        assert p["bricks"] == 1
        # a brick passes on the values of its faces only
        assert p["passed_fwd"] < n or rows < 100


def arrays(n, e):
    """1-based CSR of the pattern as csr() gives it, for large ones."""
    k = np.arange(n)
    r, c = np.concatenate([e[:, 0], e[:, 1], k]), np.concatenate([e[:, 1], e[:, 0], k])
    o = np.lexsort((c, r))
    return 1 + np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]), c[o] + 1


def test_sampled_distances():
    """A box as wide as the rows are sampled apart (every eighth of 423,200) is
    still recognised by all three distances: with parts of 64 rows a brick
    cannot hold whole lines of 8 cells in two directions."""
    assert fvk.sweep_plan(*arrays(*box(8, 230, 230)), 64)["bricks"] == 1


@pytest.mark.parametrize("holes", ["block", "cells"])
def test_irregular_boxes_are_bricks(holes):
    """Cells left out of a box shift the distances between lines and planes; a
    brick of a full box has as many rows as a part may have."""
    n, e = box(40, 40, 64)
    k = np.arange(n)
    x, y, z = k % 40, k // 40 % 40, k // 1600
    keep = ~((abs(x - 20) < 6) & (abs(y - 12) < 5) & (abs(z - 30) < 9)) if holes == "block" else k % 101 != 0
    new = np.cumsum(keep) - 1
    e = new[e[keep[e].all(1)]]
    for rows in (512, 4096):
        assert fvk.sweep_plan(*arrays(int(keep.sum()), e), rows)["bricks"] == 1


def test_choice_of_form():
    """Parts on ordered numberings; chunks where the rows are numbered at random
    and a part needs values from nearly all others."""
    n, e = box(30, 30, 30)
    parts, chunks = fvk.sweep_times(*arrays(n, e))
    assert 4 * parts < chunks
    parts, chunks = fvk.sweep_times(*arrays(n, np.random.default_rng(0).permutation(n)[e]))
    assert parts > 1.5 * chunks


@pytest.mark.parametrize("rows", [64, 300, 4096])
@pytest.mark.parametrize("n,span,width", [(50, 1, 1), (700, 3, 2), (3000, 40, 3), (3000, 3000, 4), (2000, 900, 8)])
def test_unstructured(n, span, width, rows):
    rng = np.random.default_rng(n + span)
    pairs, deg = [], np.zeros((n, 2), int)
    for i in range(1, n):
        for j in set((i - 1 - rng.integers(0, min(i, span), width)).tolist()):
            if deg[i, 0] < 8 and deg[j, 1] < 8:
                deg[i, 0] += 1
                deg[j, 1] += 1
                pairs.append((i, j))
    p = fvk.sweep_plan(*csr(n, pairs), rows)
    assert p["lds3"] <= LDS
    # the reference's loops leave entries out where columns are not sorted
    fvk.sweep_plan(*csr(n, pairs, np.random.default_rng(1)), rows)


def test_too_many_entries_is_refused():
    with pytest.raises(fvk.FvkError):
        fvk.sweep_plan(*csr(10, [(9, j) for j in range(9)]), 64)


@pytest.mark.parametrize("n,pairs", [(3000, [(i, i - 1) for i in range(1, 3000)]), box(25, 24, 23),
                                     (3000, [(i, i - j) for i in range(3000) for j in range(1, 9) if i >= j])])
def test_positions_are_limited(n, pairs):
    ia, ja = csr(n, [(int(i), int(j)) for i, j in pairs])
    p = fvk.sweep_positions(ia, ja)
    assert n <= p <= 8 * n and fvk.sweep_positions(ia, ja, limit=p) == p
    with pytest.raises(fvk.FvkError):
        fvk.sweep_positions(ia, ja, limit=p - 1)


def test_without_threads():
    """Where no thread can be started (here for want of address space for its
    stack) the calling thread does their work."""
    code = """
import resource
from programs_amd import fvk
from tests.test_sweep_plan import box, csr
n, pairs = box(40, 33, 5)
pattern = csr(n, pairs.tolist())
want = fvk.sweep_plan(*pattern, 64)
size = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (size + (256 << 20),) * 2)
assert fvk.sweep_plan(*pattern, 64) == want and want["parts"] >= 16
"""
    stack = 1 << 30
    hard = resource.getrlimit(resource.RLIMIT_STACK)[1]
    if hard != resource.RLIM_INFINITY and hard < stack:
        pytest.skip("the stack limit cannot be raised")
    subprocess.run([sys.executable, "-c", code], check=True, cwd=ROOT, timeout=120,
                   preexec_fn=lambda: resource.setrlimit(resource.RLIMIT_STACK, (stack, hard)))
