"""The neighbour search and the list walks on uneven neighbourhoods: cells from
one to the most particles a cell may hold, so that the lanes of a wavefront
find very different numbers of neighbours (rings that fill before the others
complete a group, near neighbours in several portions, lists from empty to the
longest), particle counts around a wavefront's and a block's, radii far apart
and equal.  Lists, densities, accelerations, the assembled system, gradient and
stabilisation are the oracle's bit for bit; a whole step, whose passes are
fused, assembles the system of the separate stages."""
import numpy as np
import pytest

import cases
from openmps_amd import ComputerException, _lib as L
from test_gpu_parity import compare_stage

pytestmark = pytest.mark.gpu
L0 = 0.01


def cloud(n, nl, side, cap, seed):
    """n particles in random cells of size nl (at most cap in one)."""
    rng = np.random.Generator(np.random.PCG64(seed))
    cells = rng.permutation(side * side)
    x, z, k = [], [], 0
    while len(x) < n:
        m = min(n - len(x), int(rng.integers(1, cap + 1)) if k % 3 else 1)
        c = cells[k]
        x.extend((c // side + rng.uniform(0.02, 0.98, m)) * nl)
        z.extend((c % side + rng.uniform(0.02, 0.98, m)) * nl)
        k += 1
    t = rng.choice(np.array([0, 0, 0, 0, 1, 2], np.uint8), n)
    f = [rng.standard_normal(n) * 1e-2 for _ in range(2)] + [rng.uniform(0, 100, n)]
    return dict(x=np.array(x), z=np.array(z), u=f[0], w=f[1], p=f[2], n=np.zeros(n), type=t)


@pytest.mark.parametrize("r_e,r_lap", [(2.1, 3.1), (2.4, 2.4), (3.1, 2.1)])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 255, 257, 1500])
def test_uneven_neighbourhoods(n, r_e, r_lap):
    probe = cases.make("gpu", cases.env(1e-3, 0.1, 9.8, 998.2, 1e-6, r_e, L0, 0, 0, 1, 1, r_lap), 1e-9)
    nl, cap = probe.env()["neighbor_length"], probe.grid()["cap"]
    side = max(2, int(np.ceil(np.sqrt(n / (cap / 4)))) + 1)
    env = cases.env(1e-3, 0.1, 9.8, 998.2, 1e-6, r_e, L0, 0.0, 0.0, side * nl, side * nl, r_lap)
    parts = cloud(n, nl, side, cap, 7 * n + int(10 * r_e))
    g, o, whole = cases.make("gpu", env, 1e-9), cases.make("oracle", env, 1e-9), cases.make("gpu", env, 1e-9)
    for c in (g, o, whole):
        c.add_particles(parts)
        c.set_time(1e-4, 1e-4)
    for st in ("search", "density", "error_correction", "explicit", "density", "save_x", "ppe_assemble"):
        g.stage(st)
        o.stage(st)
        compare_stage(g, o, st)
    count = g.neighbors()[0]
    print(f"  {n} particles, r {r_e}/{r_lap}: {count.min()} to {count.max()} neighbours, {cap} a cell", flush=True)
    A = g.ppe()
    for st in ("pressure_gradient", "dynamic_stabilize"):
        g.stage(st)
        o.stage(st)
        compare_stage(g, o, st)
    whole.set_time(0.0, 0.0)
    try:
        whole.forward_time(1e-4)
    except ComputerException:  # (a random cloud's system need not be solvable)
        pass
    for a, b in zip(A[:4], whole.ppe()[:4]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n,r_e,r_lap,keep", [(100_000, 2.4, 2.4, False), (100_001, 2.4, 2.4, False), (100_000, 2.1, 3.1, True),
                                              (100_001, 2.1, 3.1, True), (400_000, 2.1, 3.1, False),
                                              (400_001, 2.1, 3.1, False)])
def test_walks_chosen_by_size_and_order(n, r_e, r_lap, keep):
    """Both sides of the sizes at which the density and error-correction passes
    change their walk, in cell order and in a kept, random one."""
    probe = cases.make("gpu", cases.env(1e-3, 0.1, 9.8, 998.2, 1e-6, r_e, L0, 0, 0, 1, 1, r_lap), 1e-9)
    nl = probe.env()["neighbor_length"]
    side = int(np.ceil(np.sqrt(n) * L0 / nl)) + 1
    env = cases.env(1e-3, 0.1, 9.8, 998.2, 1e-6, r_e, L0, 0.0, 0.0, side * nl, side * nl, r_lap)
    rng = np.random.Generator(np.random.PCG64(n))
    at, w = rng.permutation(n), int(np.ceil(np.sqrt(n)))
    parts = dict(x=(at // w + 0.5 + rng.uniform(-0.3, 0.3, n)) * L0, z=(at % w + 0.5 + rng.uniform(-0.3, 0.3, n)) * L0,
                 u=rng.standard_normal(n) * 1e-2, w=rng.standard_normal(n) * 1e-2, p=rng.uniform(0, 100, n), n=np.zeros(n),
                 type=rng.choice(np.array([0, 0, 0, 0, 1, 2], np.uint8), n))
    g, o = cases.make("gpu", env, 1e-9), cases.make("oracle", env, 1e-9)
    g.set_storage_order(keep=keep)
    for c in (g, o):
        c.add_particles(parts)
        c.set_time(1e-4, 1e-4)
    for st in ("search", "density", "error_correction", "explicit", "save_x"):
        g.stage(st)
        o.stage(st)
        compare_stage(g, o, st)


@pytest.mark.parametrize("precond", [None, L.PRECOND_MULTILEVEL, L.PRECOND_AMG])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 257, 3000])
def test_fill_in_cell_and_kept_order(n, precond):
    """The assembly for particles in cell order against the general one: the same
    particles, handed over in cell order already, with the storage order kept.
    Lists, system, right-hand side and start are equal, and so are the sums that
    the preconditioners are built from: the solved pressures are equal too."""
    rng = np.random.Generator(np.random.PCG64(n))
    probe = cases.make("gpu", cases.env(1e-3, 0.1, 9.8, 998.2, 1e-6, 2.1, L0, 0, 0, 1, 1, 3.1), 1e-9)
    nl = probe.env()["neighbor_length"]
    side = int(np.ceil(np.sqrt(n) * L0 / nl)) + 1
    env = cases.env(1e-3, 0.1, 9.8, 998.2, 1e-6, 2.1, L0, 0.0, 0.0, side * nl, side * nl, 3.1)
    at = np.arange(n)
    w = int(np.ceil(np.sqrt(n)))
    parts = dict(x=(at // w + 0.5 + rng.uniform(-0.2, 0.2, n)) * L0, z=(at % w + 0.5 + rng.uniform(-0.2, 0.2, n)) * L0,
                 u=rng.standard_normal(n) * 1e-2, w=rng.standard_normal(n) * 1e-2, p=rng.uniform(0, 100, n), n=np.zeros(n),
                 type=rng.choice(np.array([0, 0, 0, 0, 1, 2], np.uint8), n))
    order = np.lexsort((at, np.floor(parts["z"] / nl), np.floor(parts["x"] / nl)))
    parts = {k: v[order] for k, v in parts.items()}
    cell, kept = cases.make("gpu", env, 1e-9), cases.make("gpu", env, 1e-9)
    kept.set_storage_order(keep=True)
    out = []
    for c in (cell, kept):
        if precond is not None:
            c.set_solver(kind=L.SOLVER_MIXED_IR, stop_rule=L.STOP_RHS_NORM, precond=precond, tol=1e-9)
        c.add_particles(parts)
        c.set_time(1e-4, 1e-4)
        for st in ("search", "density", "error_correction", "explicit", "density", "save_x", "ppe_assemble"):
            c.stage(st)
        lists, system = c.neighbors(), c.ppe()
        try:
            c.stage("ppe_solve")
        except ComputerException:  # (a cloud without a free surface need not be solvable)
            pass
        out.append((*lists, *system, c.aux("ppe_x")))
    print(f"  {n} particles: {out[0][0].max()} neighbours at most, {len(out[0][3])} entries", flush=True)
    for a, b in zip(*out):
        assert np.array_equal(a, b, equal_nan=a.dtype.kind == "f")


@pytest.mark.parametrize("height", [0.0, 0.5])
@pytest.mark.parametrize("precond", [L.PRECOND_MULTILEVEL, L.PRECOND_AMG])
def test_fill_in_a_flat_domain(precond, height):
    """A domain of no height has two rows of cells and no border above them: the
    difference of two cells' numbers does not tell which neighbours they are.
    Cell order against the kept order, as above."""
    rng = np.random.Generator(np.random.PCG64(5))
    nl = cases.make("gpu", cases.env(1e-3, 0.1, 9.8, 998.2, 1e-6, 2.1, L0, 0, 0, 1, 1, 3.1), 1e-9).env()["neighbor_length"]
    n, w = 420, 6
    env = cases.env(1e-3, 0.1, 9.8, 998.2, 1e-6, 2.1, L0, 0.0, 0.0, n // w * L0, height * nl, 3.1)
    at = np.arange(n)
    parts = dict(x=(at // w + 0.5 + rng.uniform(-0.2, 0.2, n)) * L0, z=(at % w + 0.5 + rng.uniform(-0.2, 0.2, n)) * L0,
                 u=rng.standard_normal(n) * 1e-2, w=rng.standard_normal(n) * 1e-2, p=rng.uniform(0, 100, n), n=np.zeros(n),
                 type=np.zeros(n, np.uint8))
    order = np.lexsort((at, np.floor(parts["z"] / nl), np.floor(parts["x"] / nl)))
    parts = {k: v[order] for k, v in parts.items()}
    out = []
    for keep in (False, True):
        c = cases.make("gpu", env, 1e-9)
        c.set_storage_order(keep=keep)
        assert c.grid()["nz"] == 2 + (height > 0)
        c.set_solver(kind=L.SOLVER_MIXED_IR, stop_rule=L.STOP_RHS_NORM, precond=precond, tol=1e-9)
        c.add_particles(parts)
        c.set_time(1e-4, 1e-4)
        for st in ("search", "density", "error_correction", "explicit", "density", "save_x", "ppe_assemble", "ppe_solve"):
            c.stage(st)
        out.append((c.neighbors()[0], *c.ppe(), c.aux("ppe_x"), np.array(c.solve_stats()["iterations"])))
    print(f"  {out[0][0].max()} neighbours at most, iterations {out[0][-1]} and {out[1][-1]}", flush=True)
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("nx,nz", [(1, 1), (40, 50), (61, 125), (62, 126), (128, 129), (181, 182)])
def test_cell_counts(nx, nz):
    """Grids around the size at which the scan of the cell counts goes from one
    block (8192 cells) to several launches."""
    nl = cases.make("gpu", cases.env(1e-3, 0.1, 9.8, 998.2, 1e-6, 2.1, L0, 0, 0, 1, 1, 3.1), 1e-9).env()["neighbor_length"]
    env = cases.env(1e-3, 0.1, 9.8, 998.2, 1e-6, 2.1, L0, 0.0, 0.0, nx * nl, nz * nl, 3.1)
    rng = np.random.Generator(np.random.PCG64(nx * nz))
    n = min(2000, 4 * nx * nz)
    at = rng.integers(0, nx * nz, n)
    at[-1] = nx * nz - 1  # the last cell is occupied
    zero = np.zeros(n)
    parts = dict(x=(at // nz + rng.uniform(0.02, 0.98, n)) * nl, z=(at % nz + rng.uniform(0.02, 0.98, n)) * nl, u=zero,
                 w=zero, p=zero, n=zero, type=np.zeros(n, np.uint8))
    g, o = cases.make("gpu", env, 1e-9), cases.make("oracle", env, 1e-9)
    print(f"  {g.grid()['nx']} x {g.grid()['nz']} cells", flush=True)
    for c in (g, o):
        c.add_particles(parts)
        c.stage("search")
    compare_stage(g, o, "search")


@pytest.mark.parametrize("least", [0, 15])
@pytest.mark.parametrize("most", [1, 2, 16, 17, 32, 33])
def test_cell_sizes(most, least):
    """Cells of `least` to `most` particles in random order: wavefronts whose cells all
    fit the sort's smaller network (16), that need the larger (32), that mix them,
    and cells beyond both."""
    nl = cases.make("gpu", cases.env(1e-3, 0.1, 9.8, 998.2, 1e-6, 5.0, L0, 0, 0, 1, 1, 5.0), 1e-9).env()["neighbor_length"]
    side = 13
    env = cases.env(1e-3, 0.1, 9.8, 998.2, 1e-6, 5.0, L0, 0.0, 0.0, side * nl, side * nl, 5.0)
    rng = np.random.Generator(np.random.PCG64(most))
    cells = np.repeat(np.arange(side * side), rng.integers(min(least, most), most + 1, side * side))
    cells = rng.permutation(np.append(cells, np.full(most, side * side // 2)))[:8000]
    cells = cells[np.sort(np.concatenate([np.flatnonzero(cells == c)[:most] for c in range(side * side)]))]
    n = len(cells)
    zero = np.zeros(n)
    parts = dict(x=(cells // side + rng.uniform(0.02, 0.98, n)) * nl, z=(cells % side + rng.uniform(0.02, 0.98, n)) * nl,
                 u=zero, w=zero, p=zero, n=zero, type=np.zeros(n, np.uint8))
    g, o = cases.make("gpu", env, 1e-9), cases.make("oracle", env, 1e-9)
    assert g.grid()["cap"] >= most
    print(f"  {n} particles, {np.bincount(cells).max()} in a cell at most", flush=True)
    for c in (g, o):
        c.add_particles(parts)
        c.stage("search")
    compare_stage(g, o, "search")
