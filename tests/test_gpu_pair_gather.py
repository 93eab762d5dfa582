"""The records of a wavefront's neighbours fetched together (one lane per particle): members of a batch whose size gives
every particle one lane, with fewer particles than a wavefront, whole and ragged wavefronts, empty and short lists, and
particles of many bodies, against the same members stepped alone (16 lanes each, records loaded lane by lane)."""
import numpy as np
import pytest

from opensph_amd import gpu, initial

pytestmark = pytest.mark.gpu


def member(n, seed):
    st, cfg = initial.impact(n_target=max(n, 100), n_projectile=100, r_projectile=1.5e4, offset_h=0.4, seed=seed)
    keep = np.random.default_rng(seed).permutation(st.n)[:n]
    sub = type(st)(n, st.materials)
    for k in st.a:
        sub[k][:] = st[k][keep]
    sub["flag"][:] = np.arange(n) % 40  # groups with and without a code of their own
    sub["reduce"][:] = 1.0
    sub["v"][:, :3] += np.random.default_rng(n).normal(0.0, 20.0, size=(n, 3))
    return sub, cfg


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_against_groups_of_lanes(precision):
    small = [member(n, n) for n in (1, 2, 3, 63, 64, 65, 127, 200, 1000)]
    big = initial.impact(n_target=70000, n_projectile=300, r_projectile=1.5e4, offset_h=0.4, seed=2)
    print(f"[case] pair gather {precision}", flush=True)
    alone = [gpu.GpuSolver(st, c, precision=precision) for st, c in small]
    batch = [gpu.GpuSolver(st, c, precision=precision) for st, c in small + [big]]
    for _ in range(2):
        for g in alone:
            g.dt = 1e-3
            g.step()
        for g in batch:
            g.dt = 1e-3
        gpu.step_batch(batch)
    for (st, _), a, b in zip(small, alone, batch):
        x, y = a.download(st), b.download(st)
        for k in x.a:
            assert np.array_equal(x[k], y[k]), (st.n, k)
    for g in alone + batch:
        g.close()
