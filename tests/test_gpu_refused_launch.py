"""A whole-integration launch that the device refuses: the call goes on with one launch per stage, and the
object's later launches give what they would have given.  A child process refuses a launch (a
hipLaunchKernel of its own, found before the runtime's)."""
import json
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
typedef struct { unsigned x, y, z; } grid;
int shim_count = 0, shim_refuse = -1;
int hipLaunchKernel(const void *f, grid g, grid b, void **args, size_t lds, void *stream)
{
    static int (*real)(const void *, grid, grid, void **, size_t, void *);
    if (!real) real = (int (*)(const void *, grid, grid, void **, size_t, void *))dlsym(dlopen(RUNTIME, RTLD_LAZY), "hipLaunchKernel");
    if (shim_count++ == shim_refuse) return 701;   /* hipErrorLaunchOutOfResources */
    return real(f, g, b, args, lds, stream);
}
"""

CHILD = r"""
import ctypes as C, json, sys
import numpy as np
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
from hrweno_hip import _lib
from hrweno_hip._lib import call, HrwError
count, refuse = C.c_int.in_dll(shim, "shim_count"), C.c_int.in_dll(shim, "shim_refuse")
_lib.lib()

def dev(a):
    p = C.c_void_p()
    call("hrw_device_alloc", a.nbytes, C.byref(p))
    put(p, a)
    return p
def put(p, a):
    call("hrw_memcpy_htod", p, a.ctypes.data_as(C.c_void_p), a.nbytes, None)
def get(p, n):
    a = np.empty(n)
    call("hrw_memcpy_dtoh", a.ctypes.data_as(C.c_void_p), p, a.nbytes, None)
    call("hrw_stream_synchronize", None)
    return a
def state(n):
    return 0.5 + 0.4 * np.sin(7 * (np.arange(n) + 0.5) / n)

n = 5000
u0, dt = state(n), 2e-5
prob, d, d2 = C.c_void_p(), dev(u0), dev(u0)
call("hrw_problem_burgers1d", n, 3, 1e-6, 0, 0, -1.0, -1.0, 1.0, None, 1, C.byref(prob))

# (each runs on a fresh object, `calls` times, and refuses launch `at` of the last call, counted from the
# call's first)
def refuse_at(at):
    refuse.value = count.value + at if at is not None else -1

def ode(at, calls=3):
    h = C.c_void_p()
    call("hrw_rktvd_create", prob, 3, C.byref(h))
    put(d, u0)
    t = C.c_double(0.0)
    for c in range(calls):
        refuse_at(at if c + 1 == calls else None)
        call("hrw_ode_integrate", h, d, C.byref(t), t.value + 4.5 * dt, dt, 1)
    put_back(at)
    call("hrw_ode_integrate", h, d, C.byref(t), t.value + 6.5 * dt, dt, 1)
    call("hrw_ode_destroy", h)
    return get(d, n)

def adjoint(at, calls=2):
    h = C.c_void_p()
    call("hrw_adjoint_create", prob, 3, dt, 4, 4, C.byref(h))
    for c in range(calls):
        put(d, u0)
        refuse_at(at if c + 1 == calls else None)
        call("hrw_adjoint_forward", h, d, d2)
        if at == 1:
            refuse_at(0)
        call("hrw_adjoint_backward", h, d, d)
    put_back(at)
    out = np.concatenate([get(d, n), get(d2, n)])
    call("hrw_adjoint_destroy", h)
    return out

ns = np.array([5000, 20000, 300, 9000], dtype=np.int32)
ks, dts = np.full(4, 3, dtype=np.int32), np.full(4, 1e-5)
flat = state(40000)
db = dev(flat)
def batch(at, calls=3):
    h = C.c_void_p()
    call("hrw_batch_burgers_create", 4, ns.ctypes.data_as(_lib.PI), ks.ctypes.data_as(_lib.PI), dts.ctypes.data_as(_lib.PD),
         None, None, 1e-6, 0, -1.0, 1, C.byref(h))
    put(db, flat)
    for c in range(calls):
        refuse_at(at if c + 1 == calls else None)
        call("hrw_batch_step", h, db, 70, None, 0)   # two launches, each with one behind it
    put_back(at)
    call("hrw_batch_step", h, db, 5, None, 0)
    call("hrw_batch_synchronize", h)
    out = get(db, flat.size)
    call("hrw_batch_destroy", h)
    return out

def put_back(at):
    if at is not None:
        assert count.value > refuse.value >= 0, "nothing was refused"
    refuse.value = -1

kind, ats = sys.argv[3], [int(a) for a in sys.argv[4:]]
run = {"ode": ode, "adjoint": adjoint, "batch": batch}[kind]
ref = run(None)
out = []
for at in ats:
    out.append(bool(np.array_equal(run(at), ref)))
    print(kind, "launch", at, "refused:", out[-1], file=sys.stderr, flush=True)
print(json.dumps(out))
"""


# the launches of a call in turn: a line's is the first; of a batch's 70 steps the first and the third (its
# recovery kernel follows each); an adjoint's forward and its reverse
@pytest.mark.parametrize("kind,ats", [("ode", [0]), ("adjoint", [0, 1]), ("batch", [0, 2])])
def test_refused_launches(tmp_path, kind, ats):
    runtime = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "lib", "libamdhip64.so")
    (tmp_path / "shim.c").write_text(SHIM)
    (tmp_path / "child.py").write_text(CHILD)
    so = str(tmp_path / "shim.so")
    subprocess.run(["gcc", "-shared", "-fPIC", f'-DRUNTIME="{runtime}"', "-o", so, str(tmp_path / "shim.c"), "-ldl"], check=True)
    r = subprocess.run([sys.executable, str(tmp_path / "child.py"), so, os.path.join(REPO, "hr-weno_amd"), kind, *map(str, ats)],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    assert json.loads(r.stdout.splitlines()[-1]) == [True] * len(ats), r.stderr
