"""Solves that resident workgroups give up.  One workgroup holds back before one
exchange for longer than the others wait there: those leave, it goes on as far
as their partial sums let it, and the launched kernels have to solve the
system as if nothing had run."""
import ctypes

import numpy as np
import pytest

import cases
from openmps_amd import _lib as L
from test_gpu_resident import EPS, banded

pytestmark = pytest.mark.gpu

MS = 100_000  # ticks of 10 ns


def hooks():
    lib = L.lib()
    lib.mps_drill_resident.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_int64)]
    lib.mps_resident_counts.argtypes = [ctypes.c_int] + [ctypes.POINTER(ctypes.c_int64)] * 2
    lib.mps_resident_counts.restype = None
    return lib


def drill(c, **kw):
    assert hooks().mps_drill_resident(c._h, numbers(**kw) if kw else None) == L.MPS_OK


def numbers(start=5 * MS, wait=MS, hold=20 * MS, group=0, exchange=0):
    return (ctypes.c_int64 * 5)(start, wait, hold, group, exchange)


def counts():
    a, b = ctypes.c_int64(), ctypes.c_int64()
    hooks().mps_resident_counts(0, ctypes.byref(a), ctypes.byref(b))
    return np.array([a.value, b.value])


def solved(before):
    """(ended, given up) since `before`."""
    return tuple(int(v) for v in counts() - before)


def matrix(n, reach):
    A, b, x0, _ = banded(n, reach, 9, 0, n)

    def solve(**kw):
        c = cases.make("gpu", cases.CG["env"], EPS)
        c.set_ppe(A.indptr, A.indices, A.data, b, x0)
        drill(c, **kw)
        was = counts()
        c.stage("ppe_solve")
        return c.aux("ppe_x"), c.cg_stats()["iterations"], solved(was)

    return solve, A, b, x0


@pytest.mark.parametrize("n,reach", [(700, 30), (4000, 200), (100_000, 300)])
def test_last_exchange_left_by_all_but_the_first(n, reach):
    """The first workgroup, which reports the result, finishes; the others have
    left without storing their rows of x."""
    solve, A, b, x0 = matrix(n, reach)
    x, its, how = solve()
    assert how == (1, 0)
    y, its2, how = solve(group=0, exchange=2 * its - 1)  # two exchanges an iteration
    res = np.linalg.norm(b - A @ y) / np.linalg.norm(b - A @ x0)
    print(f"  {n} rows, {its} iterations; |b - A x| / |r0| {res:.2e}", flush=True)
    assert how == (0, 1)
    # (the bound of test_gpu_resident.py)
    assert res <= 1.01 * EPS + 1e-12 * np.linalg.norm(b) / np.linalg.norm(b - A @ x0)
