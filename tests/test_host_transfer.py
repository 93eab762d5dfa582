"""copy_to_host on a runtime without a device: where results go directly, the pinned buffers and what it does when something
is not to be had."""
import pytest

import host_stub

pytestmark = pytest.mark.skipif(not host_stub.available(), reason="needs the built library and g++")


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    return host_stub.build_stub(tmp_path_factory.mktemp("stub"))


@pytest.mark.parametrize("n", [3, 2000, 300000])
def test_pinned_destination_is_copied_to_directly(stub, n):
    """A buffer that the runtime knows takes the device's copy itself: one copy of all bytes, no pinned buffer."""
    host_stub.run(stub, f"""
        s = solver({n})
        p = C.c_void_p()
        assert stub.hipHostMalloc(C.byref(p), C.c_size_t(32 * {n}), 0) == 0
        stub.stub_reset()
        assert get(s, p.value) == 0
        assert stub.stub_counter(1) == 1 and stub.stub_counter(3) == 32 * {n}, [stub.stub_counter(k) for k in range(4)]
        assert stub.stub_counter(0) == 0 and stub.stub_counter(2) == 0
    """)


def test_idle_buffers_pass_from_one_device_to_another(stub):
    """Two devices have four pinned buffers each, which is all there may be; a third one gets idle ones, with events of its
    own."""
    host_stub.run(stub, """
        out = np.zeros((300000, 4))
        for device in (0, 1, 2, 0, 2):
            stub.hipSetDevice(device)
            s = solver(300000)
            stub.stub_reset()
            assert get(s, out) == 0
            assert stub.stub_counter(0) == 0, (device, "pageable copies")
            assert stub.stub_counter(6) == 0, (device, "another device's events")
            if device == 0:
                first = s  # the pool goes with the last context
    """)


def test_no_memory_for_a_thread(stub):
    """A further copy thread whose state cannot be allocated: the calling thread does the rest."""
    host_stub.run(stub, """
        s = solver(300000)
        out = np.zeros((300000, 4))
        assert get(s, out) == 0
        stub.stub_reset()
        stub.stub_fail_new(1)
        rc = get(s, out)
        stub.stub_fail_new(0)
        assert rc == 0 and stub.stub_counter(1) == 5, (rc, stub.stub_counter(1))
    """)


def test_an_earlier_launch_error_is_reported(stub):
    """The kernel that gathers the result did not start, and no pinned buffer is to be had: the call fails all the same."""
    host_stub.run(stub, """
        s = solver(2000)
        out = np.zeros((2000, 4))
        stub.stub_fail_host_malloc(1)
        assert get(s, out) == 0  # without pinned memory
        stub.stub_fail_kernel(b"k_planes_to_stage", 1)
        assert get(s, out) != 0
        assert get(s, out) == 0  # the error was reported once
    """)
