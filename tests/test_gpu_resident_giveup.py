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


class CsrSolve:
    """mps_cg_solve_csr_noalloc on one system, or with a drill (keywords)."""

    def __init__(self, A, b, x0):
        self.hip, self.n, self.x0 = Hip(), len(b), x0
        self.args = [self.hip.put(v) for v in (A.indptr.astype(np.uint64), A.indices.astype(np.uint32), A.data, b, x0)]
        p = ctypes.c_void_p
        hooks().mps_drill_csr.argtypes = [
            ctypes.POINTER(ctypes.c_int64), ctypes.c_int, ctypes.c_size_t, p, p, p, p, p, ctypes.c_double,
            ctypes.POINTER(ctypes.c_int64), ctypes.c_char_p, ctypes.c_size_t]

    def __call__(self, **kw):
        it, err, was, x = ctypes.c_int64(-1), ctypes.create_string_buffer(256), counts(), self.args[4]
        assert self.hip.h.hipMemcpy(x, self.x0.ctypes.data, self.x0.nbytes, 1) == 0  # host to device
        if kw:
            rc = L.lib().mps_drill_csr(numbers(**kw), 0, self.n, *self.args, EPS, ctypes.byref(it), err, 256)
        else:
            rc = L.lib().mps_cg_solve_csr_noalloc(0, self.n, *self.args, EPS, 0, None, ctypes.byref(it), err, 256)
        assert rc == L.MPS_OK, err.value.decode()
        return self.hip.get(x, self.x0), it.value, solved(was)


@pytest.fixture
def csr_solves():
    """Makes CsrSolves; afterwards no refusal is remembered by the process."""
    made = []

    def make(A, b, x0):
        made.append(CsrSolve(A, b, x0))
        return made[-1]

    yield make
    for s in made:
        for _ in range(65):
            how = s()[2]
            if how != (0, 0):
                break
        s.hip.free()


@pytest.mark.parametrize("group", [0, 3])
@pytest.mark.parametrize("n,reach", [(4000, 200), (100_000, 300)])
def test_x_of_a_csr_solve_given_up(csr_solves, n, reach, group):
    A, b, x0, _ = banded(n, reach, 9, 0, n)
    solve = csr_solves(A, b, x0)
    x, its, how = solve(wait=200 * MS, hold=0)
    assert how == (1, 0)
    y, its2, how = solve(group=group, exchange=2 * its - 1)
    assert how == (0, 1)
    assert its2 == its and np.array_equal(x, y)


def test_csr_refusals_are_remembered(csr_solves):
    """After a refused system the next 1, 2, 4, ... 64 calls of its size are not
    tried, but other sizes are; after a wait that ended at its limit none of
    any size.  A resident solve ends either."""
    from test_gpu_resident_routes import one_long_row
    long, small, big = (csr_solves(*a) for a in (one_long_row(300, 140), one_long_row(301, 5), banded(4000, 200, 9, 0, 1)[:3]))
    short = csr_solves(*one_long_row(300, 5))
    ref = [s(wait=200 * MS, hold=0)[0] for s in (small, big)]
    x, _, how = long()
    assert how == (0, 1)
    for left in (1, 2, 4, 8, 16, 32, 64, 64):
        for _ in range(left):
            y, _, how = long()
            assert how == (0, 0) and np.array_equal(x, y)
        y, _, how = small()
        assert how == (1, 0) and np.array_equal(y, ref[0])
        y, _, how = long()
        assert how == (0, 1) and np.array_equal(x, y)
    for _ in range(64):
        assert short()[2] == (0, 0)
    assert short()[2] == (1, 0) and short()[2] == (1, 0)
    assert long()[2] == (0, 1) and long()[2] == (0, 0) and long()[2] == (0, 1)
    for left in (1, 2):
        y, _, how = big(group=0, exchange=0)
        assert how == (0, 1) and np.array_equal(y, ref[1])
        for k in range(left):
            y, _, how = (small, big)[k]()
            assert how == (0, 0) and np.array_equal(y, ref[k])
    assert small()[2] == (1, 0) and big()[2] == (1, 0)


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


def test_start_limit():
    """Workgroups that do not all start within the limit (none here) leave: the
    launched kernels solve, from then on for 64 solves, and after those the
    resident ones try again."""
    n = 100_000
    A, b, x0, _ = banded(n, 300, 9, 0, n)
    c = cases.make("gpu", cases.CG["env"], EPS)
    c.set_ppe(A.indptr, A.indices, A.data, b, x0)

    def solve():
        was = counts()
        c.set_aux("ppe_x", x0)
        c.stage("ppe_solve")
        return c.aux("ppe_x"), solved(was)

    x, how = solve()
    assert how == (1, 0)
    drill(c, start=0, group=1 << 20)
    y, how = solve()
    assert how == (0, 1) and np.array_equal(x, y)
    for _ in range(64):
        y, how = solve()
        assert how == (0, 0) and np.array_equal(x, y)
    y, how = solve()
    assert how == (0, 1) and np.array_equal(x, y)
    drill(c)
    y, how = solve()
    assert how == (1, 0) and np.array_equal(x, y)


def test_two_threads():
    """One resident solve at a time: a second thread's solve, while the first one
    holds back, takes the launched kernels and waits for nothing."""
    import threading
    import time
    n = 100_000
    A, b, x0, _ = banded(n, 300, 9, 0, n)
    one, two = (cases.make("gpu", cases.CG["env"], EPS) for _ in range(2))
    for c in (one, two):
        c.set_ppe(A.indptr, A.indices, A.data, b, x0)
        c.stage("ppe_solve")
        x = c.aux("ppe_x")
        c.set_aux("ppe_x", x0)
    drill(one, wait=2000 * MS, hold=300 * MS)
    was = counts()
    t = threading.Thread(target=one.stage, args=("ppe_solve",))
    t.start()
    time.sleep(0.1)  # (one's kernel runs for 0.3 s at least)
    t0 = time.perf_counter()
    two.stage("ppe_solve")
    took = time.perf_counter() - t0
    busy = t.is_alive()
    t.join()
    print(f"  the second thread's solve took {took * 1e3:.1f} ms, the first one was still running: {busy}", flush=True)
    assert solved(was) == (1, 0)
    for c in (one, two):
        assert np.array_equal(c.aux("ppe_x"), x)
