"""Results read back through the pinned pieces (2 MB, two per buffer, a further thread for every 2 MB): sizes around
whole pieces and whole shares, a stride with gaps, several threads at once; and the neighbour statistics."""
import ctypes as C
import threading

import numpy as np
import pytest

from opensph_amd import gpu, initial
from opensph_amd.state import ParticleState, RunConfig, basalt

pytestmark = pytest.mark.gpu

MB = 1 << 20


def filled(n, seed):
    st = ParticleState(n, [basalt()])
    rng = np.random.default_rng(seed)
    st["r"][:] = rng.uniform(1.0, 2.0, size=(n, 4))
    st["m"][:] = rng.random(n)
    st["flag"][:] = rng.integers(0, 1 << 30, n)
    return st


def read_back(g, st):
    n = st.n
    for field, q in (("r", "POSITION"), ("m", "MASS"), ("flag", "FLAG")):
        out = np.full_like(st[field], 7)
        g._check(g.L.osph_get_quantity(g.ctx, gpu.Q[q], 0, out.ctypes.data, 0), q)
        assert np.array_equal(out, st[field]), (n, field)
    # a stride with gaps: the bytes between the elements come back as zeros
    out = np.full((n, 6), 7.0)
    g._check(g.L.osph_get_quantity(g.ctx, gpu.Q["POSITION"], 0, out.ctypes.data, 48), "POSITION, stride 48")
    assert np.array_equal(out[:, :4], st["r"]) and not out[:, 4:].any()


@pytest.mark.parametrize("n", [0, 1, 3, MB // 32 - 1, MB // 32, MB // 32 + 1, 2 * MB // 32, 2 * MB // 32 + 1, 6 * MB // 32 + 5,
                               9 * MB // 32 - 3, 500001])
def test_sizes(n):
    st = filled(n, n)
    g = gpu.GpuSolver(st, RunConfig())
    print(f"[case] transfer n={n}", flush=True)
    read_back(g, st)
    g.close()


def test_several_threads():
    states = [filled(300000 + 17 * k, k) for k in range(6)]
    solvers = [gpu.GpuSolver(st, RunConfig()) for st in states]
    failed = []

    def work(k):
        try:
            for _ in range(5):
                read_back(solvers[k], states[k])
        except BaseException as e:  # reported below, from the test's own thread
            failed.append((k, e))

    print("[case] transfer threads", flush=True)
    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g in solvers:
        g.close()
    assert not failed, failed


@pytest.mark.parametrize("n", [1, 2, 900, 40000])
def test_neighbour_statistics(n):
    st, cfg = initial.fluid_sphere(n_requested=n, radius=500.0)
    g = gpu.GpuSolver(st, cfg)
    print(f"[case] statistics n={st.n}", flush=True)
    s = g.integrate()
    cnt = g.download(st)["ncnt"]
    assert s == dict(neighbors_min=int(cnt.min()), neighbors_max=int(cnt.max()), neighbors_mean=float(cnt.sum()) / st.n)
    stats = gpu.Stats()
    g._check(g.L.osph_integrate(g.ctx, C.byref(stats)), "again")
    assert stats.neighbors_max == cnt.max()
    g.close()
