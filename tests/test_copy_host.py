"""Host side of the field copies without a GPU: the built library over a stand-in for the HIP
runtime (hip_stub.cpp), in a process of its own.  Kernels do nothing there, so only what is
put into a field and read back, and the returned errors, mean something."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
INCLUDE = "/opt/rocm/include"

PRELUDE = """
import ctypes as C, sys
sys.path.insert(0, %r)
stub = C.CDLL(%r, mode=C.RTLD_GLOBAL)
import numpy as np
from ps3d_amd import gpu as G
def handle(*shape):
    return G.Ps3dGpu(G.make_params(*shape, extent=(1.0, 1.0, 1.0)))
def same(d, seed=1):
    for which in (G.SVORTS, G.SVOR):
        f = np.random.default_rng(seed).standard_normal((3,) + d.shape)
        d.set(which, f)
        assert np.array_equal(d.get(which), f)
SMALL, LARGE = (8, 8, 8), (128, 160, 80)     # one copy; chunks for several threads
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    from ps3d_amd import gpu
    cxx = shutil.which("g++")
    if not os.path.exists(gpu.LIB_PATH) or cxx is None or not os.path.isdir(INCLUDE):
        pytest.skip("needs the built library, g++ and the HIP headers")
    lib = str(tmp_path_factory.mktemp("stub") / "libhipstub.so")
    subprocess.run([cxx, "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I" + INCLUDE, "-o", lib,
                    os.path.join(HERE, "hip_stub.cpp")], check=True, capture_output=True)

    def go(body, **env):
        r = subprocess.run([sys.executable, "-c", PRELUDE % (ROOT, lib) + body], capture_output=True, text=True,
                           env=dict(os.environ, **env), timeout=120)
        assert r.returncode == 0, r.stderr[-2000:]
    return go


def test_fields_come_back(run):
    run("same(handle(*SMALL)); same(handle(*LARGE))")


def test_fewer_threads_where_a_buffer_cannot_be_had(run):
    """With two of eight staging buffers the copies and the calls after them go on, and the
    first missing buffer is the last one asked for."""
    run("""
d = handle(*LARGE)
same(d)
assert stub.stub_host_calls() == 2 + 4, stub.stub_host_calls()   # then one refusal in each of four copies
d.vor2vel()
""", STUB_HOST_ALLOCS="2")


def test_no_buffer_at_all_is_an_error(run):
    run("""
try:
    same(handle(*SMALL))
    raise SystemExit("no error")
except G.Ps3dError as e:
    assert "staging buffer" in str(e)
d = handle(*SMALL)
assert stub.hipGetLastError() == 0
""", STUB_HOST_ALLOCS="0")


def test_a_handle_of_another_device_than_the_current_one(run):
    """The handle's stream and the copies' events belong to its device, whichever device the
    calling thread has current; that stays current."""
    run("""
d = handle(*LARGE)
assert stub.hipSetDevice(1) == 0
same(d)
now = C.c_int()
assert stub.hipGetDevice(C.byref(now)) == 0 and now.value == 1
""")
