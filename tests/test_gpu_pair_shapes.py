"""Every launch shape of the pair kernels on states that reach it -- single lanes, groups of 4 (from 24576 particles on) and of
16 lanes, blocks of 64, 128 and 256 threads, the finalize fused or apart: a solid impact's evaluation against the oracle,
and the same bits from all shapes, alone and in batches whose members' tunings differ."""
import numpy as np
import pytest

from conftest import rel_l2
from opensph_amd import gpu
from oracle.bridge import Oracle

pytestmark = pytest.mark.gpu

DERIV = ("dv", "du", "divv", "drho", "p", "cs", "ds", "gradv", "ddamage", "reduce", "s")
SIZES = {"16 lanes": (6000, 600), "4 lanes": (28000, 2800), "single lanes": (104000, 10000)}


def impact(name):
    from cases import exercised_impact

    st, cfg = exercised_impact(*SIZES[name])
    # the lanes are chosen by these numbers
    assert {"16 lanes": st.n < 24576, "4 lanes": 24576 <= st.n < 65536, "single lanes": st.n >= 98304}[name], st.n
    return st, cfg


@pytest.fixture(scope="module", params=list(SIZES))
def case(request):
    st, cfg = impact(request.param)
    return request.param, st, cfg, Oracle().integrate(st, cfg)


SHAPES = [(lanes, block) for lanes in (1, 4) for block in (64, 128, 256)]


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-10), ("mixed", 1e-5)])
def test_an_evaluation_in_every_shape(case, precision, tol):
    name, st, cfg, want = case
    first = None
    for lanes, block in SHAPES:
        print(f"[case] pair shapes {name} n={st.n} {precision} lanes={lanes} block={block}", flush=True)
        g = gpu.GpuSolver(st, cfg, precision=precision)
        g.tune(pairs_lanes=lanes, pairs_block=block)
        g.integrate()
        got = g.download(st)
        g.close()
        if first is None:
            first = got
            assert np.array_equal(got["ncnt"], want["ncnt"])
            assert rel_l2(got["dv"][:, :3], want["dv"][:, :3]) < tol
            for k in DERIV if precision == "fp64" else ():
                assert rel_l2(got[k], want[k]) < tol, (k, rel_l2(got[k], want[k]))
        for k in got.a:
            assert np.array_equal(got[k], first[k]), (lanes, block, k)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_steps_in_every_shape(case, precision):
    name, st, cfg, _ = case
    first = None
    for fuse in (0, 1):
        for lanes, block in SHAPES:
            print(f"[case] pair shapes, steps {name} {precision} lanes={lanes} block={block} fuse={fuse}", flush=True)
            g = gpu.GpuSolver(st, cfg, precision=precision)
            g.tune(pairs_lanes=lanes, pairs_block=block, fuse_finalize=fuse)
            log = [g.step() for _ in range(2)]
            got = g.download(st)
            g.close()
            if first is None:
                first = (log, got)
            assert log == first[0]
            for k in got.a:
                assert np.array_equal(got[k], first[1][k]), (lanes, block, fuse, k)


@pytest.mark.parametrize("companion", ["4 lanes", "single lanes"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_batches_of_members_tuned_apart(companion, precision):
    """The small impact alone (16 lanes) and with a companion that decides the lanes; the members' own tunings of the lanes
    differ, and the blocks are the lead's."""
    small, large = impact("16 lanes"), impact(companion)
    alone = gpu.GpuSolver(*small, precision=precision)
    log = [alone.step() for _ in range(2)]
    want = alone.download(small[0])
    alone.close()
    for block in (64, 128, 256):
        print(f"[case] pair shapes, batch {companion} {precision} block={block}", flush=True)
        members = [gpu.GpuSolver(*s, precision=precision) for s in (small, large)]
        members[0].tune(pairs_block=block, pairs_lanes=1)
        members[1].tune(pairs_lanes=2)
        for k in range(2):
            assert members[0].dt == log[k][0]
            gpu.step_batch(members)
        assert members[0].dt == log[1][1]
        got = members[0].download(small[0])
        for g in members:
            g.close()
        for k in got.a:
            assert np.array_equal(got[k], want[k]), (block, k)
