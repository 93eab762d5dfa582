"""libosph_gpu.so on a HIP runtime without a device (hip_host_stub.cpp), in a process of its own: the library's host code
-- its pools, its plans and what it does after a failed call -- without a GPU."""
import os
import shutil
import subprocess
import sys
import textwrap

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HERE = os.path.join(ROOT, "tests")
LIB = os.path.join(ROOT, "opensph_amd", "lib", "libosph_gpu.so")

PRELUDE = f"""
import ctypes as C, sys
sys.path.insert(0, {ROOT!r})
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
stub.stub_counter.restype = C.c_longlong
stub.stub_box.argtypes = [C.c_double]
import numpy as np
from opensph_amd import gpu
from opensph_amd.state import ParticleState, RunConfig, basalt

def solver(n, precision="fp64"):
    st = ParticleState(n, [basalt()])
    st["r"][:] = np.arange(4.0 * n).reshape(n, 4)
    st["m"] = 1.0
    return gpu.GpuSolver(st, RunConfig(), precision=precision)

def get(s, out):
    return s.L.osph_get_quantity(s.ctx, gpu.Q["POSITION"], 0, out if isinstance(out, int) else out.ctypes.data, 0)
"""


def available():
    return os.path.exists(LIB) and shutil.which("g++") is not None


def build_stub(folder) -> str:
    so = os.path.join(str(folder), "libamdhip64.so.7")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-Wl,-soname,libamdhip64.so.7", "-o", so,
                    os.path.join(HERE, "hip_host_stub.cpp"), "-lpthread"], check=True)
    return so


def run(stub, body):
    """Runs `body` after the prelude (stub, solver, get) in a process of its own; fails with its output."""
    r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body), stub], capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-2000:])
    return r.stdout
