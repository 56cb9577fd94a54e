"""The particle arrays between the caller's order and the device's cell order:
every getter and setter returns and takes the caller's order whatever the
neighbour search made of it, bit for bit."""
import numpy as np
import pytest

import cases
from openmps_amd import scenes

pytestmark = pytest.mark.gpu

FIELDS = ("x", "z", "u", "w", "p", "n")


def scattered(count, seed):
    """count particles of a jittered lattice in a random order."""
    rng = np.random.Generator(np.random.PCG64(seed))
    env = cases.env(1e-3, 0.1, 9.8, 998.2, 1e-6, 2.1, 0.01, 0.0, 0.0, 1.0, 1.0, 3.1)
    side = int(np.ceil(np.sqrt(count)))
    at = rng.permutation(side * side)[:count]
    s = scenes._pack(0.1 + 0.01 * (at // side) + rng.uniform(-1e-4, 1e-4, count),
                     0.1 + 0.01 * (at % side) + rng.uniform(-1e-4, 1e-4, count),
                     rng.integers(0, 3, count).astype(np.uint8))
    return env, s, rng


@pytest.mark.parametrize("count", [1, 63, 64, 65, 257, 3001])
@pytest.mark.parametrize("searched", [False, True])
def test_state_keeps_the_callers_order(count, searched):
    print(f"  transfers: {count} particles, searched {searched}", flush=True)
    env, s, rng = scattered(count, 7 * count + searched)
    c = cases.make("gpu", env, 1e-8)
    c.add_particles(s)
    if searched:
        c.stage("search")
    got = c.particles()
    for k in FIELDS + ("type",):
        assert np.array_equal(got[k], s[k]), k
    # whole states, then single fields beside the others
    t = {k: rng.standard_normal(count) for k in FIELDS}
    t["type"] = rng.integers(0, 3, count).astype(np.uint8)
    c.set_particles(t)
    one = rng.standard_normal(count)
    c.set_particles({"p": one})
    c.set_aux("ecs", t["u"])
    got = c.particles()
    for k in FIELDS + ("type",):
        assert np.array_equal(got[k], one if k == "p" else t[k]), k
    assert np.array_equal(c.aux("ecs"), t["u"])


def test_results_in_the_callers_order():
    """Neighbour counts and densities of a shuffled scene equal those of the
    same scene kept in the caller's order."""
    env, s, _ = scattered(2500, 3)
    out = []
    for keep in (False, True):
        c = cases.make("gpu", env, 1e-8)
        c.set_storage_order(keep)
        c.add_particles(s)
        c.stage("search")
        c.stage("density")
        cnt, ids = c.neighbors()
        out.append((cnt, ids, c.particles()["n"], c.density_variation()))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("count", [1, 225, 8192, 8193])
def test_one_array_again_under_one_permutation(count):
    """The first and every later transfer of one array under a permutation, on
    both sides of the size where later ones are permuted on the host, after
    particles were added and after a new permutation."""
    print(f"  transfers again: {count} particles", flush=True)
    env, s, rng = scattered(count, 11 * count)
    first = (count + 1) // 2
    c = cases.make("gpu", env, 1e-8)
    kept = cases.make("gpu", env, 1e-8)
    kept.set_storage_order(True)
    for part in (slice(0, first), slice(first, count)):
        if part.start == part.stop:
            continue
        for m in (c, kept):
            m.add_particles({k: v[part] for k, v in s.items()})
        for _ in range(2):
            for m in (c, kept):
                m.stage("search")
                m.stage("density")
            for _ in range(3):
                assert np.array_equal(c.density_variation(), kept.density_variation())
                for a, b in zip(c.neighbors(), kept.neighbors()):
                    assert np.array_equal(a, b)
                v = rng.standard_normal(part.stop)
                c.set_aux("ecs", v)
                assert np.array_equal(c.aux("ecs"), v)
                assert np.array_equal(c.aux("ecs"), v)
            got = c.particles()
            for k in FIELDS[:4] + ("type",):
                assert np.array_equal(got[k], s[k][:part.stop]), k
