"""The host side of reading fields, on the CPU: the library runs over a HIP
runtime in host memory (csrc/host_hip.c, preloaded into a process of its own),
where a field comes back as it was uploaded."""
import os
import shutil
import subprocess
import sys

import pytest

from conftest import ROOT

HERE = os.path.dirname(os.path.abspath(__file__))

# A context of nx x ny whose fields are 4.5 MB, past the size from which several threads unpack
PROGRAM = """
import ctypes, os, sys, time
sys.path.insert(0, %r)
import numpy as np
from swm_amd import configs, gpu, host
hip = ctypes.CDLL(None)
delay = ctypes.c_int.in_dll(hip, "host_hip_thread_delay_ms")
threads = lambda: len(os.listdir("/proc/self/task"))
precision = %s
def context(nx=800, ny=700):
    s = configs.basin(nx, ny, 5e3, 5e3, variant=host.FULLY_NONLINEAR, H0=500.0, dt=5.0)
    s.u0 = np.float32(np.random.default_rng(nx).standard_normal(s.shape)).astype(float)
    s = host.finalize(s)
    return s.u0 * s.grids["u"].ocean, gpu.SwmGpu(s, precision=precision).init_from_setup()
%s
"""


@pytest.fixture(scope="module")
def host_hip(tmp_path_factory):
    if shutil.which("gcc") is None:
        pytest.skip("no C compiler")
    out = str(tmp_path_factory.mktemp("host_hip") / "libhost_hip.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", out, os.path.join(HERE, "csrc", "host_hip.c"), "-ldl",
                    "-lpthread"], check=True)
    return out


def run(host_hip, body, precision="gpu.FP64"):
    env = dict(os.environ, OMP_NUM_THREADS="1", OPENBLAS_NUM_THREADS="1")
    env["LD_PRELOAD"] = " ".join(filter(None, [host_hip, env.get("LD_PRELOAD", "")]))
    r = subprocess.run([sys.executable, "-c", PROGRAM % (ROOT, precision, body)], env=env, capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


@pytest.mark.parametrize("precision", ["gpu.FP64", "gpu.FP32"])
def test_fields_do_not_wait_for_threads_that_have_not_begun(host_hip, precision):
    """Threads that get no CPU for two seconds hold no read up, and those that
    come late find nothing left to do."""
    run(host_hip, """
u, g = context()
delay.value = 2000
t = time.perf_counter()
for _ in range(3):
    assert np.array_equal(g.get("SWM_U"), u)
assert time.perf_counter() - t < 1.0
time.sleep(2.5)
for _ in range(3):
    assert np.array_equal(g.get("SWM_U"), u)
""", precision)


def test_threads_are_few_and_end_with_the_last_context(host_hip):
    run(host_hip, """
u, g = context()
v, h = context(810, 690)
before = threads()
for _ in range(5):
    assert np.array_equal(g.get("SWM_U"), u) and np.array_equal(h.get("SWM_U"), v)
assert threads() <= before + 3
g.close()
assert np.array_equal(h.get("SWM_U"), v)
h.close()
assert threads() == before
u, g = context()
assert np.array_equal(g.get("SWM_U"), u)
g.close()
assert threads() == before
""")


def test_one_cpu_reads_without_threads(host_hip):
    run(host_hip, """
u, g = context()
before = threads()
os.sched_setaffinity(0, {min(os.sched_getaffinity(0))})
assert np.array_equal(g.get("SWM_U"), u)
assert threads() == before
""")


@pytest.mark.parametrize("nx", [800, 300])
def test_failed_wait_leaves_no_copy_into_the_staging_buffer(host_hip, nx):
    """The staging buffer is the next transfer's: a read whose wait for a piece
    fails returns only when the pieces still on their way have landed."""
    run(host_hip, """
u, g = context(%d)
assert np.array_equal(g.get("SWM_U"), u)
hip.host_hip_fail_event(2)
try:
    g.get("SWM_U")
    raise SystemExit("no error")
except gpu.SwmGpuError as e:
    assert "injected" in str(e)
assert hip.host_hip_copies_open() == 0
assert np.array_equal(g.get("SWM_U"), u)
""" % nx)
