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
from test_gpu_resident_mixed import TOL, make, scene
from test_zz_no_alloc import Hip

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


@pytest.mark.parametrize("group", [0, 3])
@pytest.mark.parametrize("n,reach", [(4000, 200), (100_000, 300)])
def test_x_of_a_solve_given_up(n, reach, group):
    """The workgroup that holds back before the last exchange stores its rows
    of x, the others do not: the launched kernels start from x as it was, and
    return what they (and the resident solve) return from there, bit for bit."""
    solve, A, b, x0 = matrix(n, reach)
    x, its, how = solve()
    assert how == (1, 0)
    y, its2, how = solve(group=group, exchange=2 * its - 1)
    assert how == (0, 1)
    assert its2 == its and np.array_equal(x, y)


@pytest.mark.parametrize("group", [0, 3])
@pytest.mark.parametrize("n,reach", [(4000, 200), (100_000, 300)])
def test_x_of_a_csr_solve_given_up(n, reach, group):
    A, b, x0, _ = banded(n, reach, 9, 0, n)
    hip = Hip()
    mat = [hip.put(A.indptr.astype(np.uint64)), hip.put(A.indices.astype(np.uint32)), hip.put(A.data), hip.put(b)]
    lib = hooks()
    p = ctypes.c_void_p
    lib.mps_drill_csr.argtypes = [ctypes.POINTER(ctypes.c_int64), ctypes.c_int, ctypes.c_size_t, p, p, p, p, p,
                                  ctypes.c_double, ctypes.POINTER(ctypes.c_int64), ctypes.c_char_p, ctypes.c_size_t]

    def solve(**kw):
        x, it, err, was = hip.put(x0), ctypes.c_int64(-1), ctypes.create_string_buffer(256), counts()
        rc = lib.mps_drill_csr(numbers(**kw), 0, n, *mat, x, EPS, ctypes.byref(it), err, 256)
        assert rc == L.MPS_OK, err.value.decode()
        return hip.get(x, x0), it.value, solved(was)

    x, its, how = solve(wait=200 * MS, hold=0)
    assert how == (1, 0)
    y, its2, how = solve(group=group, exchange=2 * its - 1)
    hip.free()
    assert how == (0, 1)
    assert its2 == its and np.array_equal(x, y)


@pytest.mark.parametrize("prec", ["ml", "amg"])
@pytest.mark.parametrize("cols,rows", [(20, 40), (127, 253)])
def test_x_of_a_refinement_given_up(prec, cols, rows):
    """Given up after at least one sweep has been added to x: the launched
    solve runs the sweeps that the resident one runs from the start."""
    def step(**kw):
        c = make(scene(cols, rows, 2.1, 3.1, False), prec)
        drill(c, **kw)
        was = counts()
        c.forward_time(1e-4)
        st = c.solve_stats()
        return c.aux("ppe_x"), [st[k] for k in ("iterations", "outer_iterations", "rr0", "rr")], solved(was)

    x, st, how = step()
    assert how == (1, 0) and st[1] >= 2
    # two exchanges an iteration (the multigrid: three at least), some more a sweep: past the first sweep, before the end
    y, st2, how = step(exchange=(2 if prec == "ml" else 3) * st[0] - 4)
    print(f"  {prec}: {st}, launched {st2}", flush=True)
    assert how == (0, 1)
    assert st2 == st and np.array_equal(x, y)
