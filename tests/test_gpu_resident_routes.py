"""Which systems the resident solvers take: both sides of each line, counted,
and the solution checked on either."""
import numpy as np
import pytest
import scipy.sparse as sp

import cases
from openmps_amd import _lib as L
from test_gpu_resident import EPS
from test_gpu_resident_giveup import counts, drill, solved
from test_gpu_resident_mixed import make, scene

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
