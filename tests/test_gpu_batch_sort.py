"""The sort by cell of all members of a batch in four launches: members whose rows of cells are empty, longer than a
wavefront or the block's LDS takes, more than a scan tile's or than its blocks' eight tiles, and tables that grow from
one step to the next, against the same members stepped alone, bit for bit."""
import numpy as np
import pytest

from opensph_amd import gpu
from opensph_amd.state import ParticleState, RunConfig, basalt

pytestmark = pytest.mark.gpu


def particles(x, h, seed, v=1.0):
    n = len(x)
    st = ParticleState(n, [basalt()])
    st["r"][:, :3] = x
    st["r"][:, 3] = h
    st["v"][:, :3] = np.random.default_rng(seed).normal(0.0, v, size=(n, 3))
    st["m"], st["rho"], st["reduce"] = 1.0, 2700.0, 1.0
    return st


def box(n, size, seed):
    return np.random.default_rng(seed).uniform(0.0, 1.0, size=(n, 3)) * np.asarray(size)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_members_equal_runs_of_their_own(precision):
    states = [
        particles(box(1, (1, 1, 1), 1), 1.0, 1),
        particles(box(6000, (3000, 1e-3, 1e-3), 2), 1.2, 2),
        particles(box(600, (300, 1e-3, 1e-3), 3), 1.2, 3),
        particles(box(5000, (1e-3, 70, 70), 4), 1.0, 4),
        particles(np.vstack([box(3000, (14, 14, 14), 5), [[0, 0, 5e4], [0, 9e4, 0], [2e5, 0, 0]]]), 1.0, 5),
        particles(np.vstack([box(1500, (13, 13, 13), 6), box(500, (4, 4, 4), 7)]),
                  np.r_[np.full(1500, 1.0), np.full(500, 0.3)], 6),
        particles(box(900, (9, 9, 9), 8), 1.0, 8, v=5e4),  # spreads: more rows every step
    ]
    cfg = RunConfig(criteria=1, initial_dt=1e-3, max_dt=1e-3)
    print(f"[case] batch sort {precision}", flush=True)
    alone = [gpu.GpuSolver(st, cfg, precision=precision) for st in states]
    batch = [gpu.GpuSolver(st, cfg, precision=precision) for st in states]
    for _ in range(4):
        for g in alone + batch:
            g.dt = 1e-3
        for g in alone:
            g.step()
        gpu.step_batch(batch)
    for k, (st, a, b) in enumerate(zip(states, alone, batch)):
        x, y = a.download(st), b.download(st)
        for f in x.a:
            assert np.array_equal(x[f], y[f]), (k, f)
    for g in alone + batch:
        g.close()
