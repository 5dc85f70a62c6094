"""The library's host code around device memory, on the CPU: libhbem.so runs on a
double of the HIP runtime (tests/cpp/hip_stub.cpp) that holds device memory in host
memory of a chosen size, can make any one allocation fail, and logs the kernel
launches instead of running them.

* A call whose allocation fails raises HBEM_ENOMEM and leaves the context as if it
  had not been made: the next call launches what a context that never failed
  launches, and holds the same device memory.
"""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes, sys
sys.path.insert(0, %r)
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
stub.hip_stub_used.restype = stub.hip_stub_peak.restype = ctypes.c_size_t
stub.hip_stub_capacity.argtypes = [ctypes.c_size_t]
stub.hip_stub_fail.argtypes = [ctypes.c_long]
stub.hip_stub_failing.restype = ctypes.c_long
stub.hip_stub_launches.restype = ctypes.c_char_p
import numpy as np
import helmholtzbem_amd as H
from helmholtzbem_amd import _lib
L = _lib.lib()
SP = H.ContinuousSpace1()
def launches():
    return stub.hip_stub_launches().decode().splitlines()
""" % ROOT


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("hip") / "libhip_stub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", out, os.path.join(HERE, "cpp", "hip_stub.cpp")],
                   check=True)
    return out


def run(stub, body):
    r = subprocess.run([sys.executable, "-c", PRELUDE + body, stub], stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-3000:]
    return r.stdout


FAILING = """
mesh = H.polygon_mesh([(0, 0), (1, 0), (1.2, 0.7), (0.1, 1)], 40)
R = H.gaussian_test_matrix(80, 2, 1)
ks = np.linspace(1.0, 9.0, 5)
calls = {
    "layers": lambda bd: H.GalerkinBuilder(bd).assembleDense(%(k)s, 2.0, H.LayerType.ALL, 2),
    "sweep": lambda bd: H.sigma_sweep(bd, ks, 1.0, 4.0, R, 2, der=2),
    "newton": lambda bd: H.sigma_sweep_der2(bd, ks, 1.0, 4.0, R, 2),
    "multi": lambda bd: H.sigma_sweep_batched([(bd, ks, 1.0, 4.0, R)], 2),
}
call = calls[%(what)r]
def steady(bd):
    H.profile_enable(bd)
    call(bd)
    launches()
    call(bd)
    return launches(), [H.profile_query(bd, w)[1:] for w in range(7)]
def builder():
    return H.BuilderData(mesh, SP, SP, 8, flags=%(flags)d)
bd = builder()
want = steady(bd)
held = stub.hip_stub_used()
failed = 0
n = 0
while True:
    n += 1
    del bd
    bd = builder()
    stub.hip_stub_fail(n)
    try:
        call(bd)
    except _lib.HbemError as e:
        assert e.code == _lib.HBEM_ENOMEM, (n, e)
        failed += 1
    else:
        assert stub.hip_stub_failing() > 0, "a failed allocation was not reported"
        stub.hip_stub_fail(0)
        break
    got = steady(bd)
    assert got == want, (n, [x for x in zip(got[0], want[0]) if x[0] != x[1]][:5], got[1], want[1])
    assert stub.hip_stub_used() == held, (n, stub.hip_stub_used(), held)
print("allocations", failed)
assert failed >= %(least)d
"""


@pytest.mark.parametrize("what,least,flags", [(w, n, f) for w, n in (("layers", 5), ("sweep", 10), ("newton", 15)) for f in (0, 1, 2)]
                         + [("multi", 3, 0), ("multi", 3, 1)])
def test_failed_allocation_leaves_no_trace(stub, what, least, flags):
    print(run(stub, FAILING % dict(what=what, least=least, flags=flags, k="3.0")))


def test_failed_allocation_leaves_no_trace_complex(stub):
    print(run(stub, FAILING % dict(what="layers", least=5, flags=0, k="3.0 + 0.05j")))


BUDGET_MULTI = """
stub.hip_stub_capacity(12 << 30)
items = []
for i in range(14):
    mesh = H.polygon_mesh([(0, 0), (1, 0), (1.2, 0.7 + 0.01 * i), (0.1, 1)], 400)
    bd = H.BuilderData(mesh, SP, SP, 8)
    items.append((bd, np.linspace(20.0, 60.0, 32), 1.0, 9.0, H.gaussian_test_matrix(800, 2, i)))
H.sigma_sweep_batched(items, 2)
launches()
first = stub.hip_stub_peak()
H.sigma_sweep_batched(items, 2)
print("device phases", sum("k_replicate_padded" in x for x in launches()), "peak", first >> 20, "MiB")
assert first <= 12 << 30
"""

BUDGET_SWEEP = """
stub.hip_stub_capacity(%(gib)d << 30)
mesh = H.polygon_mesh([(0, 0), (1, 0), (1.2, 0.7), (0.1, 1)], 600)
bd = H.BuilderData(mesh, SP, SP, 16, flags=%(flags)d)
ks = np.linspace(1.0, 40.0, 256) * %(scale)g
%(call)s
print("peak", stub.hip_stub_peak() >> 20, "MiB")
"""

SWEEP1 = "H.sigma_sweep(bd, ks, 1.0, 9.0, H.gaussian_test_matrix(1200, 2, 0), 2, der=1)"
# (without the host matrices, whose copies would be resident)
BATCH1 = "_lib.check(L.hbem_assemble_dense_batch(bd._geo.h, ks.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), 256, 9.0, 7, 1, None, None, None))"


def test_multi_sweep_budgets_its_tables(stub):
    """Fourteen instances whose tables and matrices together exceed the device: the
    tables are built before the free memory is read, so the subsets fit what is left."""
    print(run(stub, BUDGET_MULTI))


@pytest.mark.parametrize("call", [SWEEP1, BATCH1])
@pytest.mark.parametrize("what,flags,scale", [("quirk", 1, 1.0), ("beyond_the_tiers", 0, 1000.0), ("bands", 0, 1.0)])
def test_sweeps_budget_their_tables(stub, call, what, flags, scale):
    """The node tables of 180 000 panel pairs (3.3 GB) or the bands' tables are part of
    the device memory when a sweep sizes its batches."""
    print(run(stub, BUDGET_SWEEP % dict(gib=16, flags=flags, scale=scale, call=call)))
