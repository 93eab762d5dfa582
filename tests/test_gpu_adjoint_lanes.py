"""The adjoint pair sums with eight lanes to a particle: a directional derivative of one step with respect to the
initial velocities against central differences of the oracle's run, at particle counts around whole groups and blocks.

Away from the kink of the artificial viscosity at (v_i - v_j).r = 0 the final velocities are quadratic in the initial
ones, so the differences are exact there; about 1e-5 of the pairs (perturbation / velocity differences) lie at the
kink.  Rounding leaves 1e-16 * 100 / 1e-3 = 1e-11 per component."""
import numpy as np
import pytest

from opensph_amd import gpu, initial

pytestmark = pytest.mark.gpu

DT = [0.01]


@pytest.mark.parametrize("n", [10, 33, 64, 255, 257, 900])
def test_directional_derivative(n, oracle):
    st, cfg = initial.gas_collision(n_total=n, radius=1000.0, speed=100.0)
    rng = np.random.default_rng(n)
    st["v"][:, :3] += rng.normal(size=(st.n, 3)) * 100.0
    w, d = rng.normal(size=(2, st.n, 3))
    print(f"[case] adjoint lanes n={st.n}", flush=True)
    g = gpu.GpuSolver(st, cfg)
    g.adjoint_forward(DT, 1)
    grad = g.adjoint_backward(seed_v=w)["v"]
    g.close()
    eps = 1e-3
    j = []
    for s in (-eps, eps):
        moved = st.copy()
        moved["v"][:, :3] += s * d
        j.append(np.sum(oracle.run_pc_fixed(moved, cfg, DT)["v"][:, :3] * w))
    fd = (j[1] - j[0]) / (2 * eps)
    ad = np.sum(grad[:, :3] * d)
    pairs = np.linalg.norm(grad[:, :3] - w)  # what the pair sums contribute
    assert abs(ad - fd) <= (1e-4 * pairs + 1e-9 * np.linalg.norm(w)) * np.linalg.norm(d)
