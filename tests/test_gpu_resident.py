"""The solvers whose workgroups stay on the chip for the whole solve, at the
edges of what they take: one row, part-filled wavefronts and blocks, one and
two workgroups a compute unit, rows longer than the registers and the LDS
hold, unsorted columns, and systems they refuse (columns spanning too many
rows, too many rows), which the launched kernels solve."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

import cases
from openmps_amd import _lib as L
from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu

EPS = 1e-9


def say(*a):
    print(*a, flush=True)


def banded(n, reach, long_rows, far, seed):
    """A diagonally dominant symmetric system: links within `reach` rows, some
    rows with `long_rows` links, `far` links between distant rows; the entries of each row in
    random order."""
    rng = np.random.Generator(np.random.PCG64(seed))
    i, j = [], []
    for d in sorted({1, 2, max(1, reach // 2), reach}):
        if d < n:
            a = np.arange(n - d)
            a = a[rng.random(len(a)) < 0.8]
            i.append(a)
            j.append(a + d)
    for k in range(0, n, max(1, n // 7)):
        m = min(long_rows, n - 1)
        if m > 0:
            b = np.unique(np.clip(k + rng.integers(-max(reach, m), max(reach, m) + 1, m), 0, n - 1))
            i.append(np.full(len(b[b != k]), k))
            j.append(b[b != k])
    if far:
        a = rng.integers(0, n, far)
        b = (a + n // 2) % n
        i.append(a)
        j.append(b)
    i, j = (np.concatenate(v) if v else np.zeros(0, int) for v in (i, j))
    W = sp.coo_matrix((-rng.uniform(0.1, 1.0, len(i)), (i, j)), shape=(n, n)).tocsr()
    W = W + W.T
    A = (W + sp.diags(-np.asarray(W.sum(1)).ravel() + rng.uniform(0.01, 0.1, n))).tocsr()
    A.sort_indices()
    x0, b = rng.standard_normal(n), rng.standard_normal(n)
    return A, b, x0, rng


def cg(A, b, x, eps):
    """The reference CG's iterations (Computer.hpp:1382-1421) in numpy."""
    r = b - A @ x
    p = r.copy()
    rr = r @ r
    tol = eps * eps * rr
    for k in range(len(b)):
        q = A @ p
        alpha = rr / (p @ q)
        x = x + alpha * p
        r = r - alpha * q
        new = r @ r
        if new < tol:
            return x, k + 1
        p = r + (new / rr) * p
        rr = new
    return x, len(b)


SIZES = [(1, 1, 0, 0), (2, 1, 1, 0), (63, 5, 3, 0), (64, 9, 40, 0), (65, 60, 64, 0), (511, 30, 90, 0), (512, 511, 70, 0),
         (513, 100, 200, 0), (4000, 700, 35, 0), (33001, 2000, 100, 50), (131073, 1500, 40, 0), (140000, 9000, 34, 0),
         (200000, 100000, 5, 0), (262144, 300, 21, 0), (262145, 300, 21, 0)]


@pytest.mark.parametrize("n,reach,long_rows,far", SIZES)
def test_resident_cg_sizes(n, reach, long_rows, far):
    A, b, x0, rng = banded(n, reach, long_rows, far, n + reach)
    say(f"  resident CG: {n} rows, {A.nnz} entries, reach {reach}, longest row {np.diff(A.indptr).max()}")
    want, its = cg(A, b, x0, EPS)
    r0 = np.linalg.norm(b - A @ x0)
    # the caller's CSR, each row's entries in random order
    row = np.repeat(np.arange(n), np.diff(A.indptr))
    at = np.lexsort((rng.random(A.nnz), row))
    hip = Hip()
    rp, col, val = hip.put(A.indptr.astype(np.uint64)), hip.put(A.indices[at].astype(np.uint32)), hip.put(A.data[at])
    rhs = hip.put(b)
    got = []
    for _ in range(2):
        x = hip.put(x0)
        it, err = ctypes.c_int64(-1), ctypes.create_string_buffer(256)
        rc = L.lib().mps_cg_solve_csr_noalloc(0, n, rp, col, val, rhs, x, EPS, 0, None, ctypes.byref(it), err, 256)
        assert rc == L.MPS_OK, err.value.decode()
        got.append((hip.get(x, x0), it.value))
    hip.free()
    assert np.array_equal(got[0][0], got[1][0]) and got[0][1] == got[1][1]
    # and as an installed system (sliced rows, ascending columns)
    c = cases.make("gpu", cases.CG["env"], EPS)
    c.set_ppe(A.indptr, A.indices, A.data, b, x0)
    c.stage("ppe_solve")
    got.append((c.aux("ppe_x"), c.cg_stats()["iterations"]))
    for x, it in got[1:]:
        say(f"    iterations {it} (numpy {its}), |b - A x| / |r0| {np.linalg.norm(b - A @ x) / r0:.2e}")
        # the recursion's residual is below EPS |r0|; the true one differs by rounding, n u |A||x| at most here
        assert np.linalg.norm(b - A @ x) <= 1.01 * EPS * r0 + 1e-12 * np.linalg.norm(b)
        assert abs(it - its) <= max(2, 0.02 * its)


@pytest.mark.parametrize("n", [100, 600])
def test_resident_cg_iteration_limit(n):
    """A limit below the iterations needed is reported as the launched kernels
    report it, after exactly that many iterations."""
    from openmps_amd import ComputerException
    A, b, x0, _ = banded(n, 7, 3, 0, 5)
    _, its = cg(A, b, x0, EPS)
    c = cases.make("gpu", cases.CG["env"], EPS)
    c.set_ppe(A.indptr, A.indices, A.data, b, x0)
    c.set_solver(tol=EPS, max_iter=its // 2)
    with pytest.raises(ComputerException):
        c.stage("ppe_solve")
    assert c.cg_stats()["iterations"] == its // 2
