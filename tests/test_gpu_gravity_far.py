"""Two clusters so far apart that the squared distance between them overflows: the attraction across is zero, and every
particle keeps that of its own cluster."""
import numpy as np
import pytest

from opensph_amd.gravity import G_SI, GpuGravity
from oracle.bridge import GravityOracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver,leaf", [("barnes_hut", 25), ("barnes_hut", 64), ("barnes_hut", 4), ("brute_force", 25)])
@pytest.mark.parametrize("kernel", ["m4", "point"])
def test_separations_past_the_square_root_of_the_largest_number(solver, leaf, kernel):
    rng = np.random.default_rng(3)
    near = rng.uniform(-1.0, 1.0, size=(20, 3))
    far = 1.0e160 * np.array([1.0, 0.2, -0.3]) + 1.0e150 * rng.uniform(-1.0, 1.0, size=(20, 3))
    r = np.c_[np.vstack([near, far]), np.full(40, 0.3)]
    m = rng.uniform(1.0, 2.0, 40)
    print(f"[case] far clusters {solver} {kernel} leaf {leaf}", flush=True)
    g = GpuGravity(r, m, theta=0.5, order="monopole", leaf_size=leaf, kernel=kernel, solver=solver)
    g.build()
    a, _ = g.eval_self()
    g.close()
    want = GravityOracle().direct(r[:20], m[:20], G_SI, kernel=kernel)
    # 20 terms of at most the largest pull each, rounded by a few units of 2^-53; the tree's own nodes (leaf 4) come with
    # their expansion's error
    assert np.all(np.isfinite(a))
    assert np.array_equal(a[20:], np.zeros((20, 3)))
    assert np.max(np.abs(a[:20] - want)) <= (1e-13 if leaf >= 20 else 0.3) * np.max(np.abs(want))
