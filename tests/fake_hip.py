"""The HIP stand-in (fake_hip.c) for child processes that test the host
driver's error paths: `run(body)` runs Python code in one, with `fake` the
stand-in, `abi` the bindings over it, `graph(E)` an uploaded graph and `pend()`
the launches and copies nobody has waited for."""
import os
import subprocess
import sys
import tempfile

TESTS = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(TESTS)
_so = None

HEAD = """
import ctypes, os, sys
fake = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)
fake.fake_used.restype = fake.fake_peak.restype = ctypes.c_size_t
fake.fake_trace.restype = ctypes.c_char_p
fake.fake_limit.argtypes = [ctypes.c_size_t]
fake.fake_pairs.argtypes = [ctypes.c_ulonglong]
fake.fake_steal_ticks.restype = ctypes.c_longlong
sys.path[:0] = [%r, %r]
import numpy as np
from everest_amd import abi
from oracle import prep
from helpers import random_graph
assert abi.lib().tm_device_count() == 1

def graph(E=500, N=40):
    U, V, T = random_graph(np.random.default_rng(E), E, N, 4 * E)
    return abi.DeviceGraph.from_dict(prep.preprocess(U, V, T))

def fails(call, status=None):
    try:
        call()
    except abi.TMError as e:
        assert status is None or e.status == status, e
        return e
    raise AssertionError("did not fail")

pend = fake.fake_pending
MOT = [(0, 1, 0), (1, 2, 1), (2, 0, 2)]
"""


def library():
    global _so
    if _so is None:
        _so = os.path.join(tempfile.mkdtemp(prefix="fakehip"), "libfakehip.so")
        subprocess.check_call(["gcc", "-O1", "-shared", "-fPIC", "-w", "-I/opt/rocm/include",
                               "-I" + os.path.join(ROOT, "everest_amd", "csrc", "hip"),
                               os.path.join(TESTS, "fake_hip.c"), "-o", _so])
    return _so


def run(body):
    env = dict(os.environ, OMP_NUM_THREADS="2")
    p = subprocess.run([sys.executable, "-c", HEAD % (library(), ROOT, TESTS) + body], env=env, timeout=100,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, cwd=ROOT)
    assert p.returncode == 0, "exit %d\n%s" % (p.returncode, p.stdout[-3000:])
    return p.stdout
