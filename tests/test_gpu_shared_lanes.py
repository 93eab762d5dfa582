"""Groups of lanes that share a particle in the list kernel (below 131072 particles) and the pair kernels (16 lanes
below 24576 particles, 4 below 65536): counts that leave the last wavefront ragged and counts on both sides of the
rules, against the oracle; and the same bits from a group as from a single lane."""
import dataclasses

import numpy as np
import pytest

from opensph_amd import gpu, initial
from oracle.bridge import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 5, 70, 1000, 23000, 23200, 61500, 62000, 122500, 124500])
def test_evaluation_against_the_oracle(n):
    """One derivative evaluation: FP64 at the parity bar 1e-10, mixed precision at its bar 1e-5."""
    st, cfg = initial.fluid_sphere(n_requested=n, radius=500.0, sigma_v=5.0, seed=n)
    print(f"[case] shared lanes n={st.n}", flush=True)
    want = Oracle().integrate(st, cfg)
    for precision, tol in (("fp64", 1e-10), ("mixed", 1e-5)):
        g = gpu.GpuSolver(st, cfg, precision=precision)
        g.integrate()
        got = g.download(st)
        g.close()
        assert np.array_equal(got["ncnt"], want["ncnt"])
        for k in ("dv", "drho", "du"):
            a, b = got[k], want[k]
            assert np.linalg.norm(a - b) <= tol * max(np.linalg.norm(b), np.finfo(float).tiny), (precision, k)


@pytest.mark.parametrize("companion", [30000, 64000])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_a_group_of_lanes_makes_the_sums_of_one(precision, companion):
    """A small solid impact and a small fluid sphere stepped alone (16 lanes per particle) and in a batch with a
    larger companion (4 lanes, or one): every quantity bit for bit."""
    impact, cfg = initial.impact(n_target=2600, n_projectile=300, r_projectile=1.5e4, offset_h=0.4, seed=5)
    impact["v"][:, :3] += np.random.default_rng(1).normal(0.0, 20.0, size=(impact.n, 3))
    fluid, fcfg = initial.fluid_sphere(n_requested=1500, radius=500.0, sigma_v=5.0, seed=3)
    big, bcfg = initial.fluid_sphere(n_requested=companion, radius=2000.0, sigma_v=5.0, seed=4)
    assert (big.n >= 65536) == (companion == 64000) and big.n >= 24576
    print(f"[case] group of lanes, {precision}, companion {big.n}", flush=True)
    small = [(impact, dataclasses.replace(cfg, initial_dt=1e-3)), (fluid, fcfg)]
    alone = [gpu.GpuSolver(st, c, precision=precision) for st, c in small]
    batch = [gpu.GpuSolver(st, c, precision=precision) for st, c in small + [(big, bcfg)]]
    for _ in range(4):
        for g in alone:
            g.step()
        gpu.step_batch(batch)
    for (st, _), a, b in zip(small, alone, batch):
        assert a.dt == b.dt
        x, y = a.download(st), b.download(st)
        for k in x.a:
            assert np.array_equal(x[k], y[k]), k
    assert np.any(alone[0].download(impact)["gradv"] != 0.0)
    for g in alone + batch:
        g.close()
