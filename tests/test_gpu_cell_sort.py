"""The sort by cell through rows of cells: pair sets bit-identical to the oracle's and a repeatable order where the
rows are empty, short, longer than a wavefront takes (512 particles) and longer than the block's LDS takes (2048),
with several smoothing-length classes and with far outliers that stretch the grid to its 250 cells per axis."""
import numpy as np
import pytest

from opensph_amd import gpu
from opensph_amd.state import ParticleState, RunConfig, basalt
from oracle.bridge import Oracle

pytestmark = pytest.mark.gpu


def particles(x, h, seed):
    n = len(x)
    st = ParticleState(n, [basalt()])
    st["r"][:, :3] = x
    st["r"][:, 3] = h
    st["v"][:, :3] = np.random.default_rng(seed).normal(0.0, 1.0, size=(n, 3))
    st["m"] = 1.0
    st["rho"] = 2700.0
    st["reduce"] = 1.0
    return st


def box(n, size, seed):
    return np.random.default_rng(seed).uniform(0.0, 1.0, size=(n, 3)) * np.asarray(size)


CASES = {
    "one": lambda: (box(1, (1, 1, 1), 1), 1.0),
    "line along x": lambda: (box(6000, (3000, 1e-3, 1e-3), 2), 1.2),
    "short line": lambda: (box(600, (300, 1e-3, 1e-3), 3), 1.2),
    "line along z": lambda: (box(6000, (1e-3, 1e-3, 3000), 4), 1.2),
    "sheet": lambda: (box(5000, (70, 70, 1e-3), 5), 1.0),
    "outliers": lambda: (np.vstack([box(3000, (14, 14, 14), 6), [[0, 0, 5e4], [0, 9e4, 0], [2e5, 0, 0]]]), 1.0),
    "outliers and classes": lambda: (np.vstack([box(2500, (13, 13, 13), 7), box(1500, (4, 4, 4), 8), [[-3e3, 0, 0]]]),
                                     np.r_[np.full(2500, 1.0), np.full(1500, 0.3), [4.1]]),
    "lattice": lambda: (np.stack(np.meshgrid(*[np.arange(17.0)] * 3, indexing="ij"), -1).reshape(-1, 3), 1.0),
}


@pytest.mark.parametrize("name", list(CASES))
def test_pair_sets_and_order(name):
    x, h = CASES[name]()
    st = particles(x, h, 11)
    cfg = RunConfig(criteria=1, initial_dt=1e-6)
    print(f"[case] cell sort {name} n={st.n}", flush=True)
    want = np.stack(Oracle().pairs(st["r"]), axis=1)
    want = want[np.lexsort((want[:, 1], want[:, 0]))]
    runs = []
    for precision in ("fp64", "mixed", "fp64"):
        g = gpu.GpuSolver(st, cfg, precision=precision)
        assert np.array_equal(np.stack(g.pairs(), axis=1), want)
        # a second search from the state in cell order, and the derivatives it gives
        g.integrate()
        g.integrate()
        runs.append(g.download(st))
        g.close()
    for k in ("dv", "drho", "du", "ncnt"):
        assert np.array_equal(runs[0][k], runs[2][k]), k
