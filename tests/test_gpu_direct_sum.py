"""The direct sum with the terms of a chunk of 64 sources shared by the wavefronts of a block of 16 targets: the terms
and their order are the oracle's (compiled without contraction), so are the sums, bit for bit, at sizes around whole
chunks and blocks, for pairs inside and outside the softening, and where a term leaves the form for ordinary pairs."""
import numpy as np
import pytest

from opensph_amd.gravity import GpuGravity
from oracle.bridge import GravityOracle

pytestmark = pytest.mark.gpu

G = 6.674e-11


def particles(n, seed, scale=1.0, grid=False):
    rng = np.random.default_rng(seed)
    r = rng.normal(size=(n, 4))
    if grid:  # equal coordinates: separations with zero components, no coincident particles
        side = int(np.ceil(n ** (1 / 3)))
        k = np.arange(n)
        r[:, :3] = np.stack([k % side, k // side % side, k // side ** 2], 1)
    r[:, 3] = rng.uniform(0.05, 0.4, n)
    return r * scale, rng.uniform(0.5, 2.0, n) * 1e20


@pytest.mark.parametrize("kernel", ["m4", "point"])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 64, 65, 128, 1000, 4097])
def test_sizes(n, kernel):
    r, m = particles(n, n)
    print(f"[case] direct n={n} {kernel}", flush=True)
    g = GpuGravity(r, m, solver="brute_force", kernel=kernel, G=G)
    g.build()
    a, _ = g.eval_self()
    assert np.array_equal(a[:, :3], GravityOracle().direct(r, m, G, kernel=kernel))
    for nt in (1, 15, 17):
        pick = np.random.default_rng(nt).integers(0, n, nt).astype(np.uint32)
        assert np.array_equal(g.direct(pick)[:, :3], a[pick, :3])


# coordinates whose squares, cubes and quotients leave the bounds of the ordinary form (and of FP64), and lattices
@pytest.mark.parametrize("kernel", ["m4", "point"])
@pytest.mark.parametrize("scale, grid", [(1e-145, False), (1e-52, False), (1e-45, False), (1e47, False), (1e53, False),
                                         (1e99, False), (1.0, True), (1e6, True)])
def test_ranges(scale, grid, kernel):
    r, m = particles(300, 5, scale, grid)
    print(f"[case] direct scale={scale} grid={grid} {kernel}", flush=True)
    g = GpuGravity(r, m, solver="brute_force", kernel=kernel, G=G)
    g.build()
    a, _ = g.eval_self()
    ref = GravityOracle().direct(r, m, G, kernel=kernel)
    assert np.array_equal(a[:, :3], ref, equal_nan=True)
