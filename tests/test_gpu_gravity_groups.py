"""The Barnes-Hut walk over groups of targets and the sums of their lists at the sizes where the groups, the lane
splits and the lists are ragged: one to a few particles, leaves of one and of 64 particles, a last group that is
not full, targets shared by a block and targets of their own, lists that outgrow their first capacity.  At theta
-> 0 every leaf is summed pair by pair, so the result is the direct sum."""
import numpy as np
import pytest

from opensph_amd.gravity import G_SI, GpuGravity
from oracle.bridge import GravityOracle

pytestmark = pytest.mark.gpu


def ball(n, seed):
    rng = np.random.default_rng(seed)
    x = rng.normal(size=(n, 3))
    x *= (1.0e4 * rng.random(n) ** (1 / 3) / np.linalg.norm(x, axis=1))[:, None]
    return np.c_[x, rng.uniform(100.0, 900.0, n)], rng.uniform(0.5, 2.0, n) * 1e12


@pytest.mark.parametrize("n,leaf", [(1, 1), (2, 1), (3, 25), (26, 25), (65, 64), (129, 64), (700, 1), (1001, 13),
                                    (3001, 1)])
@pytest.mark.parametrize("kernel", ["m4", "point"])
def test_sums_at_theta_zero_equal_the_direct_sum(n, leaf, kernel):
    r, m = ball(n, n + leaf)
    print(f"[case] groups n={n} leaf={leaf} {kernel}", flush=True)
    want = GravityOracle().direct(r, m, G_SI, kernel=kernel)
    top = max(np.max(np.abs(want)), np.finfo(float).tiny)
    for precision, tol in (("fp64", 8.0 * n * 2.0 ** -53), ("mixed", 1e-6)):
        g = GpuGravity(r, m, kernel=kernel, theta=1e-12, order=2, leaf_size=leaf, precision=precision)
        g.build()
        a, st = g.eval_self()
        g.close()
        assert st["pairs"] == n * (n - 1) and st["expansions"] == 0
        assert np.max(np.abs(a - want)) <= max(tol, 1e-15) * top


@pytest.mark.parametrize("n,leaf,order", [(40009, 25, 2), (130003, 17, 3)])
def test_shared_and_own_targets_against_sampled_direct_sums(n, leaf, order):
    """Fewer targets than a block each takes, and more: theta -> 0 against the direct sum of 300 particles, and
    theta 0.5 with equal counts and sums on both sides of the FP32 screen."""
    r, m = ball(n, n)
    pick = np.random.default_rng(n).choice(n, 300, replace=False).astype(np.uint32)
    print(f"[case] groups shared n={n} leaf={leaf}", flush=True)
    g = GpuGravity(r, m, theta=1e-12, order=order, leaf_size=leaf)
    g.build()
    a, st = g.eval_self()
    want = g.direct(pick)
    g.close()
    assert st["pairs"] == n * (n - 1)
    assert np.max(np.abs(a[pick] - want)) <= 8.0 * n * 2.0 ** -53 * np.max(np.abs(want))
    out = []
    for screen in (0, 1):
        g = GpuGravity(r, m, theta=0.5, order=order, leaf_size=leaf)
        g.tune(walk_screen=screen)
        g.build()
        out.append(g.eval_self())
        g.close()
    assert out[0][1] == out[1][1] and np.array_equal(out[0][0], out[1][0])
