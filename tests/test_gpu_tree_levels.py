"""Node moments where depths of few nodes go through one block: root moments against the oracle's direct ones (1e-10, as
for the tree as a whole) around runs of 256 nodes, in bushy trees and in thin, deep ones; and a wait for the host's words
that outlasts the watch of 20 ms."""
import dataclasses

import numpy as np
import pytest

from opensph_amd import gpu, initial
from opensph_amd.gravity import G_SI, GpuGravity
from oracle.bridge import GravityOracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", ["cloud", "line"])
@pytest.mark.parametrize("n", [2, 3, 200, 257, 513, 3000])
def test_root_moments(n, shape):
    rng = np.random.default_rng(n)
    r = np.ones((n, 4))
    r[:, :3] = rng.uniform(-1.0, 1.0, (n, 3))
    if shape == "line":  # every halving of the range leaves a few particles behind
        r[:, :3] = 2.0 ** (-20.0 * np.arange(n) / n)[:, None]
    r[:, 3] = 0.01
    m = rng.uniform(1.0, 2.0, n)
    print(f"[case] levels n={n} {shape}", flush=True)
    g = GpuGravity(r, m, theta=0.5, order=3, leaf_size=1, G=1.0)
    g.build()
    got, want = g.moments(), GravityOracle().moments(r, m)
    assert got[0] == pytest.approx(want[0], rel=1e-10)
    assert np.max(np.abs(got[1:4] - want[1:4])) <= 1e-10 * np.max(np.abs(r[:, :3]))
    assert np.max(np.abs(got[4:] - want[4:])) <= 1e-10 * np.abs(want[4:]).max() + 1e-12


def test_long_wait():
    """The direct sum of 120k particles takes some 40 ms before the neighbour lists of the same evaluation."""
    st, cfg = initial.gas_collision(n_total=120000, radius=1000.0, speed=100.0)
    print(f"[case] long wait n={st.n}", flush=True)
    g = gpu.GpuSolver(st, cfg)
    g.integrate()
    alone = g.download(st)["dv"].copy()
    g.close()
    g = gpu.GpuSolver(st, dataclasses.replace(cfg, gravity=1))
    g.integrate()
    both = g.download(st)["dv"]
    g.close()
    d = GpuGravity(st["r"], st["m"], solver="brute_force", G=G_SI)
    d.build()
    own, _ = d.eval_self()
    # the pair sums follow on the gravity: rounding of 50 terms of the size of the accelerations
    rest = both[:, :3] - alone[:, :3] - own[:, :3]
    assert np.max(np.abs(rest)) <= 50 * 1.2e-16 * np.max(np.abs(alone)) + 1e-14 * np.max(np.abs(own))
    assert np.max(np.abs(rest)) <= 1e-6 * np.max(np.abs(own))
