"""Particles of infinite, undefined and vanishing mass or density in the pair sums: a term that a pair does not have adds
nothing, whatever the factors, so infinities and NaN end up where a single lane, and the oracle, have them."""
import numpy as np
import pytest

from opensph_amd import gpu
from oracle.bridge import Oracle

pytestmark = pytest.mark.gpu

FIELDS = ("dv", "du", "divv", "drho", "gradv", "ds")


def kinds(x):
    """0 for a number, 1 for NaN, 2 and 3 for the infinities."""
    x = np.asarray(x)
    return np.where(np.isnan(x), 1, np.where(np.isposinf(x), 2, np.where(np.isneginf(x), 3, 0)))


def impact(field, value):
    from cases import exercised_impact

    st, cfg = exercised_impact(2500, 250)
    for i in (5, st.n // 2):
        st[field][i] = value
    return st, cfg


@pytest.mark.parametrize("field,value", [("m", np.inf), ("m", -np.inf), ("m", np.nan), ("m", 0.0), ("rho", np.inf),
                                         ("rho", 1e-320), ("u", np.nan), ("m", 1e300)])
def test_an_evaluation_has_them_where_the_oracle_has(field, value):
    st, cfg = impact(field, value)
    print(f"[case] odd values, {field} = {value}", flush=True)
    with np.errstate(all="ignore"):
        want = Oracle().integrate(st, cfg)
    g = gpu.GpuSolver(st, cfg)
    g.integrate()
    got = g.download(st)
    g.close()
    for k in FIELDS:
        assert np.array_equal(kinds(got[k]), kinds(want[k])), (k, np.argwhere(kinds(got[k]) != kinds(want[k]))[:5])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("field,value", [("m", np.inf), ("m", np.nan), ("rho", np.inf)])
def test_any_lanes_give_the_same(field, value, precision):
    """The step of a small impact (16 lanes) with a companion that makes it 4 lanes, or one.  The search before it grows
    the neighbour lists, as a member whose lists overflow in a batch ends the step alone."""
    from cases import exercised_impact

    st, cfg = impact(field, value)
    alone = gpu.GpuSolver(st, cfg, precision=precision)
    alone.pairs()
    alone.dt = 1e-9
    alone.step()
    want = alone.download(st)
    alone.close()
    for size in ((28000, 2800), (104000, 10000)):
        print(f"[case] odd values, {precision} {field} = {value}, companion {size}", flush=True)
        members = [gpu.GpuSolver(*s, precision=precision) for s in ((st, cfg), exercised_impact(*size))]
        for g in members:
            g.pairs()
            g.dt = 1e-9
        gpu.step_batch(members)
        got = members[0].download(st)
        for g in members:
            g.close()
        for k in got.a:
            assert np.array_equal(got[k], want[k], equal_nan=True), k
