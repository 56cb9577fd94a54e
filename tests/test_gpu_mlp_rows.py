"""The training kernels at the edges of their tiles: rows around a K step of the
products (64), the rows of a block of the activations' backward (32), one and
several parts of a weight gradient, against the oracle's formulas with the
kernels' BF16 roundings.  What is left is FP32 summation (1e-6) and values that
round to the other BF16 neighbour because of it: at most one in a hundred by
2^-8, 4e-4 in the norm; one row too many or too few in 8193 would be 1e-2."""
import numpy as np
import pytest

from oracle import mlp as omlp
from test_mlp import FEAT, random_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 31, 33, 63, 64, 65, 127, 257, 1000, 4095, 8193])
def test_gradients_row_counts(rows):
    from openmps_amd.learned import Model
    p = random_params(5)
    m = Model(0)
    m.set_params(p)
    rng = np.random.Generator(np.random.PCG64(rows))
    x = omlp.to_bf16(rng.normal(size=(rows, FEAT)))
    t = rng.normal(size=rows).astype(np.float32).astype(np.float64)
    w1, w2 = omlp.to_bf16(p["w1"]), omlp.to_bf16(p["w2"])
    z1 = x @ w1.T + p["b1"]
    h1 = omlp.to_bf16(omlp.gelu(z1))
    a2 = h1 @ w2.T + p["b2"]
    h2 = omlp.gelu(a2)
    y = h2 @ p["w3"] + p["b3"][0]
    dy = 2 * (y - t) / rows
    da2 = dy[:, None] * p["w3"] * omlp.gelu_grad(a2)
    da2b = omlp.to_bf16(da2)
    da1 = (da2b @ w2) * omlp.gelu_grad(z1)
    want = {"w1": omlp.to_bf16(da1).T @ x, "b1": da1.sum(0), "w2": da2b.T @ h1, "b2": da2.sum(0), "w3": h2.T @ dy,
            "b3": np.array([dy.sum()])}
    for _ in range(2):  # (the second call finds the first one's buffers)
        loss, g = m.gradients(x, t)
        assert abs(loss - np.mean((y - t) ** 2)) <= 1e-4 * np.mean((y - t) ** 2)
        for k in want:
            err = np.linalg.norm(g[k] - want[k]) / np.linalg.norm(dy) / max(1.0, np.linalg.norm(want[k]) / np.linalg.norm(dy))
            print(f"  {rows} rows, {k}: {err:.1e}", flush=True)
            assert err <= 1e-3, (k, err)


def test_rows_that_no_memory_holds():
    """A call whose buffers cannot be allocated (2^40 rows; nothing is read)
    fails, and the next calls work: fewer rows than before it, and more."""
    from openmps_amd import _lib as L
    from openmps_amd.learned import Model
    m = Model(0)
    m.set_params(random_params(5))
    rng = np.random.Generator(np.random.PCG64(1))
    x = rng.normal(size=(600, FEAT)).astype(np.float32)
    t = rng.normal(size=600).astype(np.float32)
    y, (loss, g) = m.forward(x[:300]), m.gradients(x[:300], t[:300])
    few = np.zeros(4, np.float32)
    assert L.lib().mps_model_forward(m._h, 1 << 40, few.ctypes.data, few.ctypes.data) == L.MPS_ERR_HIP
    assert np.array_equal(m.forward(x[:300]), y) and np.array_equal(m.forward(x[:200]), y[:200])
    loss2, g2 = m.gradients(x[:300], t[:300])
    assert abs(loss2 - loss) <= 1e-5 * loss  # (its atomics add in any order)
    for k in g:
        assert np.linalg.norm(g2[k] - g[k]) <= 1e-5 * np.linalg.norm(g[k])
    assert np.array_equal(m.forward(x)[:300], y)
