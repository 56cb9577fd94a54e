"""The mixed multilevel and multigrid solvers with resident workgroups (a
scene's own solve) against the launched kernels (the same scene in a batch):
scenes at the edges of what the resident solve takes: a few cells, one block
of rows, a level held in LDS or spread over the workgroups, one and two
workgroups a compute unit, more than that, wide radii; limited sweeps; a
target that FP32 sweeps cannot meet.

Both solves meet |b - A p| <= TOL |b|, so in the first step, from the same
state and system, |A (p - p')| <= 2 TOL |b|.  The two run the same
iterations; their FP64 residual norms are summed in different orders, which
can move a stop test by one iteration of a sweep."""
import numpy as np
import pytest
import scipy.sparse

from openmps_amd import Batch, Computer, _lib as L, make_environment, scenes

pytestmark = pytest.mark.gpu
TOL = 1e-10
PREC = {"ml": L.PRECOND_MULTILEVEL, "amg": L.PRECOND_AMG}


def scene(cols, rows, r_e, r_lap, still):
    l0 = 1e-3
    tank = cols * l0 if still else 3 * cols * l0
    parts, dom = scenes.dam_break(tank, 1.2 * rows * l0, cols * l0, rows * l0, l0, 0.02, cols)
    env = make_environment(dict(max_dt=1e-4, courant=0.1, g=9.8, rho=998.2, nu=1.004e-6, r_e_by_l0=r_e, l0=l0,
                                r_lap_by_l0=r_lap, **dom))
    return env, parts


def make(sc, prec, **kw):
    c = Computer(1e-10, sc[0])
    c.set_solver(kind=L.SOLVER_MIXED_IR, stop_rule=L.STOP_RHS_NORM, precond=PREC[prec], tol=TOL, **kw)
    c.add_particles(sc[1])
    return c


def solved(c):
    rp, col, val, b, x = c.ppe()
    return scipy.sparse.csr_matrix((val, col.astype(np.int64), rp.astype(np.int64)), shape=(len(b),) * 2), b, x


# columns, rows, radii, column as wide as the tank
SHAPES = [(2, 3, 2.1, 3.1, False), (3, 5, 2.1, 3.1, True), (11, 20, 3.1, 3.1, False), (16, 16, 2.4, 2.4, True),
          (50, 101, 2.4, 2.4, True), (61, 117, 2.1, 3.1, False), (130, 200, 2.1, 2.1, True), (127, 253, 2.1, 3.1, False),
          (260, 400, 3.1, 3.1, True), (250, 480, 2.1, 3.1, True), (300, 600, 2.1, 3.1, False), (400, 700, 2.1, 2.4, True)]


@pytest.mark.parametrize("prec", ["ml", "amg"])
@pytest.mark.parametrize("cols,rows,r_e,r_lap,still", SHAPES)
def test_resident_and_launched(prec, cols, rows, r_e, r_lap, still):
    sc = scene(cols, rows, r_e, r_lap, still)
    own, other = make(sc, prec), make(sc, prec)
    batch = Batch([other])
    own.forward_time(1e-4)
    batch.forward_time(1e-4)
    a, b = own.solve_stats(), other.solve_stats()
    A, rhs, x = solved(own)
    A2, rhs2, x2 = solved(other)
    assert np.array_equal(A.data, A2.data) and np.array_equal(rhs, rhs2)
    diff = np.linalg.norm(A @ (x - x2)) / max(np.linalg.norm(rhs), 1e-300)
    print(f"  {prec} {own.size()} particles: {a['iterations']} iterations in {a['outer_iterations']} sweeps, launched "
          f"{b['iterations']} in {b['outer_iterations']}; |A (p - p')| / |b| {diff:.2e}", flush=True)
    assert a["rel_residual"] <= TOL and b["rel_residual"] <= TOL
    assert np.linalg.norm(rhs - A @ x) <= 1.01 * TOL * np.linalg.norm(rhs)
    assert diff <= 2.02 * TOL
    assert a["outer_iterations"] == b["outer_iterations"]
    assert abs(a["iterations"] - b["iterations"]) <= a["outer_iterations"]


@pytest.mark.parametrize("prec", ["ml", "amg"])
@pytest.mark.parametrize("cols,rows", [(20, 40), (127, 253)])
def test_limited_sweeps(prec, cols, rows):
    """Sweeps of at most 5 iterations: each takes exactly 5 until the last."""
    sc = scene(cols, rows, 2.1, 3.1, False)
    c = make(sc, prec, inner_max_iter=5)
    c.forward_time(1e-4)
    st = c.solve_stats()
    A, rhs, x = solved(c)
    assert np.linalg.norm(rhs - A @ x) <= 1.01 * TOL * np.linalg.norm(rhs)
    assert st["fallback"] or 5 * (st["outer_iterations"] - 1) < st["iterations"] <= 5 * st["outer_iterations"]


@pytest.mark.parametrize("prec", ["ml", "amg"])
def test_target_below_rounding(prec):
    """A target that no FP64 residual meets: the sweeps stall and the plain CG
    finishes by its recursion's residual (the reference's stop rule)."""
    sc = scene(20, 40, 2.1, 3.1, False)
    c = make(sc, prec)
    c.set_solver(kind=L.SOLVER_MIXED_IR, stop_rule=L.STOP_RHS_NORM, precond=PREC[prec], tol=1e-25)
    c.forward_time(1e-4)
    st = c.solve_stats()
    assert st["fallback"] == 1 and st["outer_iterations"] >= 3


@pytest.mark.parametrize("prec", ["ml", "amg"])
@pytest.mark.parametrize("cols,rows", [(20, 40), (127, 253)])
def test_fallback_is_part_of_the_solve(prec, cols, rows):
    """The plain CG that finishes a stalled refinement: its time is in solve_ms,
    and the refinement holds nothing that keeps it from running resident."""
    c = make(scene(cols, rows, 2.1, 3.1, False), prec)
    c.set_solver(kind=L.SOLVER_MIXED_IR, stop_rule=L.STOP_RHS_NORM, precond=PREC[prec], tol=1e-25)
    c.set_profiling(True)
    c.forward_time(1e-4)
    st, k = c.solve_stats(), c.kernel_stats()
    # both are launches between the solve's two events
    inside = k["cg_spmv32"]["ms"] + k["cg_spmv"]["ms"]
    print(f"  {prec}: solve {st['solve_ms']:.3f} ms, its kernels {inside:.3f} ms, launches {k['cg_spmv']['launches']}",
          flush=True)
    assert st["fallback"] == 1
    assert st["solve_ms"] >= inside
    assert k["cg_spmv"]["launches"] == 1 and k["cg_update"]["launches"] == 0


@pytest.mark.parametrize("warm", ["previous", "learned"])
@pytest.mark.parametrize("prec", ["ml", "amg", "auto"])
@pytest.mark.parametrize("cols,rows", [(5, 9), (60, 117), (300, 600)])
def test_solver_chosen_after_the_search(cols, rows, prec, warm):
    """A search under the FP64 solver lists no blocks of cells for the
    preconditioners: the set-up of the first mixed solve does, on the auxiliary
    stream if the learned start runs before it, and the solve has to wait for
    their number.  Same system, same solver: the same bits as with the solver
    chosen first, in the first solve and in a second one."""
    from openmps_amd import learned
    model = learned.Model(3)

    def run(late):
        sc = scene(cols, rows, 2.1, 3.1, False)
        c = Computer(1e-10, sc[0])
        c.add_particles(sc[1])
        learned.attach_model(c, model)

        def choose():
            c.set_solver(kind=L.SOLVER_MIXED_IR, stop_rule=L.STOP_RHS_NORM, tol=TOL,
                         precond=dict(PREC, auto=L.PRECOND_AUTO)[prec],
                         warm_start=L.WARM_LEARNED if warm == "learned" else L.WARM_PREVIOUS)

        if not late:
            choose()
        c.set_time(1e-4, 1e-4)
        for stage in ("search", "density", "error_correction", "explicit", "density"):
            c.stage(stage)
        if late:
            choose()
        out = []
        for _ in range(2):
            c.stage("ppe_assemble")
            c.stage("ppe_solve")
            st = c.solve_stats()
            assert st["rel_residual"] <= TOL
            out.append((c.aux("ppe_x"), st["iterations"], st["precond_used"]))
        return out

    early, late = run(False), run(True)
    print(f"  {prec} {warm}: {[v[1:] for v in early]}, chosen late {[v[1:] for v in late]}", flush=True)
    if prec == "auto":  # (its second choice follows the times of the first)
        early, late = early[:1], late[:1]
    for (x, it, used), (x2, it2, used2) in zip(early, late):
        assert it == it2 and used == used2 and np.array_equal(x, x2)


@pytest.mark.parametrize("prec", ["ml", "amg", "auto"])
@pytest.mark.parametrize("cols,rows", [(5, 9), (60, 117), (300, 600)])
def test_solver_chosen_after_the_assembly(cols, rows, prec):
    """The system assembled under the FP64 solver, which sums no rows for the
    preconditioners: set-up and block list come with the solve.  The sums are
    taken in another order, which can move a stop test by one iteration of a
    sweep (as above)."""
    def run(late):
        sc = scene(cols, rows, 2.1, 3.1, False)
        c = Computer(1e-10, sc[0])
        c.add_particles(sc[1])
        opts = dict(kind=L.SOLVER_MIXED_IR, stop_rule=L.STOP_RHS_NORM, tol=TOL, precond=dict(PREC, auto=L.PRECOND_AUTO)[prec])
        if not late:
            c.set_solver(**opts)
        c.set_time(1e-4, 1e-4)
        for stage in ("search", "density", "error_correction", "explicit", "density", "ppe_assemble"):
            c.stage(stage)
        if late:
            c.set_solver(**opts)
        c.stage("ppe_solve")
        A, rhs, x = solved(c)
        assert np.linalg.norm(rhs - A @ x) <= 1.01 * TOL * np.linalg.norm(rhs)
        return c.solve_stats()

    a, b = run(False), run(True)
    print(f"  {prec}: {a['iterations']} iterations in {a['outer_iterations']} sweeps, {b['iterations']} in "
          f"{b['outer_iterations']}", flush=True)
    assert a["precond_used"] == b["precond_used"] and a["outer_iterations"] == b["outer_iterations"]
    assert abs(a["iterations"] - b["iterations"]) <= a["outer_iterations"]
