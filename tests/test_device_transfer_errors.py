"""The entry points that take the caller's device memory wait for the work they
queued on every return, whichever of their HIP calls fails
(include/des_amd.h: "the context's stream is synchronized on return"): a
caller frees or reuses its tensors after an error too.

On the CPU: a process of its own in which tests/hip_stub.c takes the HIP
runtime's place and fails the calls one after the other."""
import os
import subprocess
import sys

import pytest

from dynearthsol_amd import lib

HERE = os.path.dirname(os.path.abspath(__file__))
pytestmark = pytest.mark.skipif(not os.path.exists(lib.LIB_PATH), reason="library not built")

PROGRAM = r"""
import ctypes as C, sys
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)     # ahead of the HIP runtime in the lookup order
stub.stub_left.restype = C.c_long
stub.stub_fail_at.argtypes = [C.c_long]
sys.modules["torch"] = None
sys.path[:0] = sys.argv[2:4]
import numpy as np
import scenarios as SC
from dynearthsol_amd import model as M
from dynearthsol_amd.lib import DesError, DesModel

def each_failure(make, call):
    n = failed = 0
    while True:
        g = make()
        a = {k: np.zeros(6 * g.E) for k in ("coord", "vel", "temperature", "stress", "plstrain", "elem_visc", "elem_cohesion")}
        p = {k: v.ctypes.data for k, v in a.items()}
        g.sync()
        assert stub.stub_pending() == 0
        stub.stub_fail_at(n)
        try:
            call(g, p)
            error = None
        except DesError as ex:
            error = ex
            failed += 1
        reached = stub.stub_left() < 0
        stub.stub_fail_at(-1)
        assert not stub.stub_pending(), "call %d failed (%s): returned with work queued" % (n, error)
        g.close()
        if not reached:
            assert error is None and failed > 1, (n, failed, error)
            return failed
        assert error is not None, "call %d failed and nothing was reported" % n
        n += 1

small = SC.build("evp3", nelem=300)
adjoint = M.config_adjoint("maxwell", nelem_target=300)
plain = lambda: DesModel(small, init=False)

def recorded():
    g = DesModel(adjoint, init=False)
    g.upload(elem_visc=np.full(g.E, 1e22), elem_cohesion=np.full(g.E, 4e7))
    g.adj_forward(2, 0)
    return g

print("upload", each_failure(plain, lambda g, p: g.upload_device(**p)))
print("download", each_failure(plain, lambda g, p: g.download_device(**{k: p[k] for k in ("coord", "vel", "stress")})))
print("backward", each_failure(recorded, lambda g, p: g.adj_backward_device(p["coord"], p["elem_visc"], p["elem_cohesion"])))
"""


def test_every_failing_call_is_waited_for(tmp_path):
    stub = str(tmp_path / "libhip_stub.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-w", os.path.join(HERE, "hip_stub.c"), "-o", stub], check=True)
    r = subprocess.run([sys.executable, "-c", PROGRAM, stub, os.path.dirname(HERE), HERE], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stderr[-2000:]
