"""Objects that find no memory for what only the whole-integration launches need are created all the
same and give the same results by one launch per stage.  A child process refuses one allocation of an
object after the other (a hipMalloc of its own, found before the runtime's)."""
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
int shim_count = 0, shim_refuse = -1;
int hipMalloc(void **p, size_t n)
{
    static int (*real)(void **, size_t);
    if (!real) real = (int (*)(void **, size_t))dlsym(dlopen(RUNTIME, RTLD_LAZY), "hipMalloc");
    if (shim_count++ == shim_refuse) {
        *p = NULL;
        return 2;   /* hipErrorOutOfMemory */
    }
    return real(p, n);
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

def ode(handle=None):
    if handle is None:
        h = C.c_void_p()
        call("hrw_rktvd_create", prob, 3, C.byref(h))
        return h
    put(d, u0)
    t = C.c_double(0.0)
    call("hrw_ode_integrate", handle, d, C.byref(t), 4.5 * dt, dt, 1)
    call("hrw_ode_destroy", handle)
    return get(d, n)

def adjoint(handle=None):
    if handle is None:
        h = C.c_void_p()
        call("hrw_adjoint_create", prob, 3, dt, 4, 4, C.byref(h))
        return h
    put(d, u0)
    call("hrw_adjoint_forward", handle, d, d2)
    call("hrw_adjoint_backward", handle, d, d)
    out = np.concatenate([get(d, n), get(d2, n)])
    call("hrw_adjoint_destroy", handle)
    return out

ns = np.array([5000, 20000, 300, 9000], dtype=np.int32)
ks, dts = np.full(4, 3, dtype=np.int32), np.full(4, 1e-5)
flat = state(40000)
db = dev(flat)
def batch(handle=None):
    if handle is None:
        h = C.c_void_p()
        call("hrw_batch_burgers_create", 4, ns.ctypes.data_as(_lib.PI), ks.ctypes.data_as(_lib.PI), dts.ctypes.data_as(_lib.PD),
             None, None, 1e-6, 0, -1.0, 1, C.byref(h))
        return h
    put(db, flat)
    call("hrw_batch_step", handle, db, 3, None, 0)
    call("hrw_batch_synchronize", handle)
    out = get(db, flat.size)
    call("hrw_batch_destroy", handle)
    return out

make = {"ode": ode, "adjoint": adjoint, "batch": batch}[sys.argv[3]]
before = count.value
handle = make()
total = count.value - before
ref = make(handle)
went = []
for i in range(total):
    refuse.value = count.value + i
    try:
        handle = make()
    except HrwError as e:
        assert e.code == 3, e
        continue
    finally:
        refuse.value = -1
    went.append(bool(np.array_equal(make(handle), ref)))
    print(sys.argv[3], "allocation", i, "of", total, "refused:", went[-1], file=sys.stderr, flush=True)
print(json.dumps({"total": total, "went": went}))
"""


@pytest.mark.parametrize("kind,optional", [("ode", 1), ("adjoint", 2), ("batch", 3)])
def test_refused_allocations(tmp_path, kind, optional):
    runtime = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "lib", "libamdhip64.so")
    (tmp_path / "shim.c").write_text(SHIM)
    (tmp_path / "child.py").write_text(CHILD)
    so = str(tmp_path / "shim.so")
    subprocess.run(["gcc", "-shared", "-fPIC", f'-DRUNTIME="{runtime}"', "-o", so, str(tmp_path / "shim.c"), "-ldl"], check=True)
    r = subprocess.run([sys.executable, str(tmp_path / "child.py"), so, os.path.join(REPO, "hr-weno_amd"), kind],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    out = json.loads(r.stdout.splitlines()[-1])
    assert out["total"] > optional and all(out["went"]) and len(out["went"]) == optional, (out, r.stderr)
