"""Plans whose allocations fail: the call says so, nothing is left half made, and
the next call with memory to be had works from the start.  Runs the library's
host code over a HIP runtime of its own (hip_host.cpp), without a GPU."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

DRIVER = r'''
import ctypes, sys
host = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
for f in ('host_allocations', 'host_live', 'host_launches'):
    getattr(host, f).restype = ctypes.c_long
host.host_fail_at.argtypes = [ctypes.c_long]
mode, precondition = int(sys.argv[2]), int(sys.argv[3])
import numpy as np
from gpaw_amd import _lib
from gpaw_amd.fd_operators import Laplace
from gpaw_amd.grid_descriptor import GridDescriptor
from gpaw_amd.transformers import Transformer
L = _lib.lib()
gd = [GridDescriptor((32, 32, 32), (8, 8, 8), True)]
while len(gd) < 3:
    gd.append(gd[-1].coarsen())
ops = [Laplace(g, -0.25 / np.pi, 3 if i == 0 else 1) for i, g in enumerate(gd)]
rst = [Transformer(a, b, 1) for a, b in zip(gd, gd[1:])]
itp = [Transformer(b, a, 1) for a, b in zip(gd, gd[1:])]
VP = ctypes.c_void_p

def new(h):
    return L.gpaw_poisson_new(
        2, (VP * 3)(*[o.operator.h for o in ops]), (VP * 2)(*[t.transformer.h for t in rst]),
        (VP * 2)(*[t.transformer.h for t in itp]), (ctypes.c_int * 3)(2, 4, 8),
        (ctypes.c_int * 3)(1, 4, 8), (ctypes.c_double * 3)(2 / 3, 1, 1), 2, gd[0].dv,
        ctypes.byref(h))

def plan():
    h = VP()
    _lib.check(new(h))
    return h

a, b = np.zeros((32,) * 3), np.zeros((32,) * 3)

def solve(h):
    if mode < 0:     # the FP64 solver; no kernel runs, so the charge and errors are zero
        q, err = ctypes.c_double(0), ctypes.c_double(0)
        neutral, niter = ctypes.c_int(0), ctypes.c_int(0)
        return L.gpaw_poisson_solve(h, a.ctypes.data, b.ctypes.data, 1e-10, 50, 1e-6,
                                    ctypes.byref(q), ctypes.byref(neutral), ctypes.byref(niter),
                                    ctypes.byref(err), None)
    if precondition:
        return L.gpaw_poisson_precondition(h, a.ctypes.data, b.ctypes.data, mode >> 1, None)
    niter, rel = ctypes.c_int(0), ctypes.c_double(0)
    return L.gpaw_poisson_solve_mixed(h, a.ctypes.data, b.ctypes.data, 1e-10, 50, mode, 1,
                                      ctypes.byref(niter), ctypes.byref(rel), None)

first = plan()           # what the operators keep is made here
assert solve(first) == 0
L.gpaw_poisson_free(first)
empty = host.host_live()
host.host_fail_at(0)
h = plan()
made = host.host_live()
for n in range(1, host.host_allocations() + 1):
    host.host_fail_at(n)
    assert new(VP()) != 0 and host.host_live() == made, n
host.host_fail_at(0)
assert solve(h) == 0
needed, whole = host.host_allocations(), host.host_live()
assert needed > 5 and whole > made
L.gpaw_poisson_free(h)
assert host.host_live() == empty
for n in range(1, needed + 1):
    h = plan()
    host.host_fail_at(n)
    rc = solve(h)
    assert rc != 0, n
    host.host_fail_at(0)
    rc = solve(h)
    assert rc == 0, (n, rc)
    assert host.host_live() == whole, (n, host.host_live(), whole)
    L.gpaw_poisson_free(h)
    assert host.host_live() == empty, n
print('allocations', needed, 'ok')
'''


@pytest.fixture(scope='module')
def shim(tmp_path_factory):
    so = str(tmp_path_factory.mktemp('hip') / 'libhiphost.so')
    subprocess.run(['g++', '-O1', '-shared', '-fPIC', os.path.join(HERE, 'hip_host.cpp'), '-o', so],
                   check=True)
    return so


@pytest.mark.parametrize('precondition', [0, 1])
@pytest.mark.parametrize('mode', [1, 3, 0])
def test_mixed_solver_after_a_failed_allocation(shim, mode, precondition):
    """mode: CG with the FP32 and with the FP64 inner V-cycle, refinement."""
    r = subprocess.run([sys.executable, '-c', DRIVER, shim, str(mode), str(precondition)],
                       cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().endswith('ok'), r.stdout + r.stderr


def test_fp64_solver_after_a_failed_allocation(shim):
    r = subprocess.run([sys.executable, '-c', DRIVER, shim, '-1', '0'], cwd=ROOT,
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().endswith('ok'), r.stdout + r.stderr
