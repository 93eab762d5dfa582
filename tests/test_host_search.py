"""A neighbour search whose launches fail, on a runtime without a device: the calls after it start from clean row counts, and
nothing is launched on what the failed kernel did not write."""
import pytest

import host_stub

pytestmark = pytest.mark.skipif(not host_stub.available(), reason="needs the built library and g++")

BODY = """
    s = solver(64, {precision!r})
    def call():
        nd, crit, dt = C.c_double(), C.c_int(), 1e-6
        if {batch}:
            two = (C.c_void_p * 2)(s.ctx, other.ctx)
            return s.L.osph_step_pc_batch(two, 2, (C.c_double * 2)(dt, dt), (C.c_double * 2)(), (C.c_int * 2)())
        return s.L.osph_step_pc(s.ctx, dt, C.byref(nd), C.byref(crit))
    other = solver(64, {precision!r})
    for g in (s, other):
        g.tune(sort_cells={cells}, batch_graph=0)
    stub.stub_box(30.0)
    assert call() == 0
    stub.stub_reset()
    assert call() == 0 and stub.stub_counter(5) == {scatters}
    stub.stub_fail_kernel({kernel!r}, 1)
    assert call() != 0
    assert stub.stub_counter(8) == 0, "launches after the failed one"
    stub.stub_reset()
    for _ in range(2):
        assert call() == 0
    assert stub.stub_counter(4) == 0, "row counts that do not start at zero"
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    return host_stub.build_stub(tmp_path_factory.mktemp("stub"))


@pytest.mark.parametrize("kernel", ["k_row_count", "k_row_scan", "k_row_scatter", "k_row_order"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_a_failed_launch_of_the_sort(stub, kernel, precision):
    host_stub.run(stub, BODY.format(precision=precision, batch=False, cells=0, scatters=1, kernel=kernel.encode()))


@pytest.mark.parametrize("kernel", ["k_fill_u32", "k_row_count", "k_row_scan", "k_cell_starts", "k_row_scatter", "k_cell_order"])
def test_a_failed_launch_of_the_sort_by_cells(stub, kernel):
    host_stub.run(stub, BODY.format(precision="fp64", batch=False, cells=1, scatters=1, kernel=kernel.encode()))


@pytest.mark.parametrize("cells,kernel", [(0, "kb_row_scatter"), (1, "kb_cell_clear"), (1, "kb_cell_starts"), (0, "kb_row_order"), (0, "kb_lists")])
def test_a_failed_launch_in_a_batch(stub, cells, kernel):
    host_stub.run(stub, BODY.format(precision="fp64", batch=True, cells=cells, scatters=0, kernel=kernel.encode()))


def test_a_batch_has_no_limit_of_the_grid(stub):
    """The members lie along x, whose extent is 2^31 - 1 blocks; y and z end at 65535."""
    host_stub.run(stub, """
        members = [solver(64) for _ in range(5)]
        for g in members:
            g.tune(batch_graph=0)
        stub.stub_reset()
        ctxs = (C.c_void_p * 5)(*[g.ctx for g in members])
        assert members[0].L.osph_step_pc_batch(ctxs, 5, (C.c_double * 5)(*[1e-6] * 5), (C.c_double * 5)(), (C.c_int * 5)()) == 0
        assert stub.stub_counter(7) == 1, stub.stub_counter(7)
    """)


@pytest.mark.parametrize("lanes", [(1, 1), (1, 2), (4, 1), (2, 4)])
def test_members_with_other_lanes_are_batched(stub, lanes):
    """The sums are the same bits whatever the lanes per particle, so these do not keep members apart."""
    host_stub.run(stub, f"""
        members = [solver(64) for _ in range(2)]
        for g, lanes in zip(members, {lanes}):
            g.tune(pairs_lanes=lanes)
        stub.stub_reset()
        ctxs = (C.c_void_p * 2)(*[g.ctx for g in members])
        assert members[0].L.osph_step_pc_batch(ctxs, 2, (C.c_double * 2)(1e-6, 1e-6), (C.c_double * 2)(), (C.c_int * 2)()) == 0
        assert stub.stub_counter(9) > 0
    """)


def test_the_tuner_times_every_launch_shape_once(stub):
    """The default space, in the library and in Python: no two candidates that are the same launch at every size."""
    host_stub.run(stub, """
        from opensph_amd import autotune
        s = solver(64)
        trials = C.c_int()
        chosen = (C.c_longlong * 5)()
        best = C.c_double()
        assert s.L.osph_step_pc(s.ctx, 1e-6, None, None) == 0
        assert s.L.osph_autotune(s.ctx, 1e-6, 1, None, None, None, 0, chosen, C.byref(best), None, 0, C.byref(trials)) == 0
        assert trials.value == 1 + sum(len(v) - 1 for _, v in autotune.DEFAULT_SPACE)
        lanes = dict(autotune.DEFAULT_SPACE)["pairs_lanes"]
        assert len(lanes) == len({4 if v > 1 else 1 for v in lanes})  # 2 and 4 are one launch
    """)


@pytest.mark.parametrize("call", ["osph_integrate(s.ctx, None)", "osph_step_pc(s.ctx, 1e-6, None, None)", "osph_build_neighbors(s.ctx)"])
def test_a_failed_launch_of_the_lists(stub, call):
    """The pair sums would follow entries that nobody wrote."""
    host_stub.run(stub, f"""
        s = solver(64)
        assert s.L.{call} == 0
        stub.stub_reset()
        stub.stub_fail_kernel(b"k_neighbor_lists", 1)
        assert s.L.{call} != 0
        assert stub.stub_counter(8) == 0, stub.stub_counter(8)
        assert s.L.{call} == 0
    """)


@pytest.mark.parametrize("kernel", ["k_morton", "k_radix_tree", "k_mark_leaves", "k_depth"])
def test_a_failed_launch_of_the_tree(stub, kernel):
    """The moments index by depths and children."""
    host_stub.run(stub, f"""
        from opensph_amd.gravity import GpuGravity
        g = GpuGravity(np.arange(256.0).reshape(64, 4), np.ones(64))
        assert g.L.osph_gravity_build(g.ctx) == 0
        stub.stub_reset()
        stub.stub_fail_kernel({kernel.encode()!r}, 1)
        assert g.L.osph_gravity_build(g.ctx) != 0
        assert stub.stub_counter(8) == 0, stub.stub_counter(8)
        assert g.L.osph_gravity_build(g.ctx) == 0
    """)
