"""Which systems the resident solvers take: both sides of each line, counted,
the solution checked on either, and the same bits from the launched kernels."""
import numpy as np
import pytest
import scipy.sparse as sp

import cases
from openmps_amd import _lib as L
from test_gpu_resident import EPS, SIZES, banded
from test_gpu_resident_giveup import counts, drill, solved
from test_gpu_resident_mixed import SHAPES, make, scene

pytestmark = pytest.mark.gpu


def one_long_row(n, m):
    """A chain of n rows whose first row has m off-diagonal entries."""
    rng = np.random.Generator(np.random.PCG64(n + m))
    i = np.concatenate([np.arange(1, n - 1), np.zeros(m, int)])
    j = np.concatenate([np.arange(2, n), np.arange(1, m + 1)])
    W = sp.coo_matrix((-rng.uniform(0.1, 1.0, len(i)), (i, j)), shape=(n, n)).tocsr()
    W = W + W.T
    A = (W + sp.diags(-np.asarray(W.sum(1)).ravel() + rng.uniform(0.01, 0.1, n))).tocsr()
    A.sort_indices()
    return A, rng.standard_normal(n), rng.standard_normal(n)


# one workgroup a compute unit: 32 entries in registers, 26 in LDS (144 KB less 12 KB of marks and the list of rows,
# 5 KB an entry of 512 rows), 24 streamed; two: 20, 11 and 18
@pytest.mark.parametrize("n,m,resident", [(300, 82, True), (300, 83, False), (300, 140, False), (600, 250, False),
                                          (140_000, 49, True), (140_000, 50, False), (140_000, 400, False)])
def test_long_rows(n, m, resident):
    A, b, x0 = one_long_row(n, m)
    c = cases.make("gpu", cases.CG["env"], EPS)
    c.set_ppe(A.indptr, A.indices, A.data, b, x0)
    was = counts()
    c.stage("ppe_solve")
    how = solved(was)
    x = c.aux("ppe_x")
    r0 = np.linalg.norm(b - A @ x0)
    print(f"  {n} rows, the longest of {m}: (ended, given up) {how}", flush=True)
    assert how == ((1, 0) if resident else (0, 1))
    assert np.linalg.norm(b - A @ x) <= 1.01 * EPS * r0 + 1e-12 * np.linalg.norm(b)  # (as test_gpu_resident.py)


@pytest.mark.parametrize("profiling", [False, True])
@pytest.mark.parametrize("prec", ["ml", "amg"])
@pytest.mark.parametrize("cols,rows", [(20, 40), (127, 253)])
def test_bytes_of_a_resident_refinement(prec, cols, rows, profiling):
    """The kernel statistics account for a resident refinement, one launch, the
    bytes that they account for the launched kernels of the same solve (given up
    at its first exchange, then launched)."""
    kernels = ("cg_spmv32", "ml_prec", "amg_cycle", "cg_init32", "ir_residual")

    def step(**kw):
        c = make(scene(cols, rows, 2.1, 3.1, False), prec)
        drill(c, **kw)
        c.set_profiling(profiling)
        c.reset_kernel_stats()
        was = counts()
        c.forward_time(1e-4)
        k = c.kernel_stats()
        return sum(k[name]["bytes"] for name in kernels), k["cg_spmv32"]["launches"], solved(was)

    own, launches, how = step()
    assert how == (1, 0) and launches == 1
    launched, launches, how = step(exchange=0)
    print(f"  {prec}: {own:.6e} bytes, launched {launched:.6e}", flush=True)
    assert how == (0, 1) and launches > 1
    assert own == pytest.approx(launched, rel=1e-12)


def both_ways(make_context, run):
    """A solve as it comes, and by the launched kernels (given up at its first
    exchange; a drill has no shape for two workgroups a compute unit)."""
    out = []
    for kw in ({}, dict(exchange=0)):
        c = make_context()
        drill(c, **kw)
        was = counts()
        run(c)
        st = c.solve_stats()
        out.append((solved(was), c.aux("ppe_x"), [st[k] for k in ("iterations", "outer_iterations", "rr0", "rr")]))
    return out


# workgroups of 512 rows on the 256 compute units, one or two on each
ONE, TWO = 131_072, 262_144


@pytest.mark.parametrize("n,reach,long_rows,far", SIZES)
def test_systems_resident_and_launched(n, reach, long_rows, far):
    """Bit for bit the same, and resident where rows and spans fit (above)."""
    A, b, x0, _ = banded(n, reach, long_rows, far, n + reach)
    longest = np.diff(A.indptr).max() - 1
    first, last = A.indices[A.indptr[:-1]], A.indices[A.indptr[1:] - 1]  # (sorted rows)
    span = max(last[k:k + 512].max() - first[k:k + 512].min() for k in range(0, n, 512))
    resident = n <= TWO and span < 65536 and longest <= (82 if n <= ONE else 49)

    def context():
        c = cases.make("gpu", cases.CG["env"], EPS)
        c.set_ppe(A.indptr, A.indices, A.data, b, x0)
        return c

    (how, x, st), (how2, x2, st2) = both_ways(context, lambda c: c.stage("ppe_solve"))
    print(f"  {n} rows, longest {longest}, span {span}: (ended, given up) {how} and {how2}, {st}", flush=True)
    assert how == ((1, 0) if resident else (0, 1) if n <= TWO else (0, 0))
    assert how2 != (1, 0) or n <= 512  # (a single workgroup waits for no other)
    assert st == st2 and np.array_equal(x, x2)


@pytest.mark.parametrize("prec", ["ml", "amg"])
@pytest.mark.parametrize("cols,rows,r_e,r_lap,still", SHAPES)
def test_scenes_resident_and_launched(prec, cols, rows, r_e, r_lap, still):
    """Bit for bit the same; resident up to one workgroup a compute unit (multigrid) or two."""
    sc = scene(cols, rows, r_e, r_lap, still)
    (how, x, st), (how2, x2, st2) = both_ways(lambda: make(sc, prec), lambda c: c.forward_time(1e-4))
    print(f"  {prec} {len(x)} particles: (ended, given up) {how} and {how2}, {st}", flush=True)
    assert how == ((1, 0) if len(x) <= (ONE if prec == "amg" else TWO) else (0, 0))
    assert how2 != (1, 0) or len(x) <= 512
    assert st == st2 and np.array_equal(x, x2)
