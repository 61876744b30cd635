"""FAST reconstructions at the ends of the range of numbers: each face is the quotient that the host's
division gives (the same header compiled for the host), to jumps whose products overflow; where products
underflow (faces below 1e-240), to two ulp: the quotient's one correction may be lost there, which
leaves the roundings of the reciprocal and of the product."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MATH = os.path.join(REPO, "hr-weno_amd", "csrc", "weno_math.hpp")

PROGRAM = f"""
#include "{MATH}"
template <int K> static void run(long n, const double *v, double eps, double *vl, double *vr)
{{
    for (long i = 0; i < n; ++i) {{
        double x[2 * K - 1];
        for (int m = -(K - 1); m <= K - 1; ++m) {{
            const long j = i + m;
            x[m + K - 1] = v[j < 0 ? 0 : (j >= n ? n - 1 : j)];
        }}
        hrw::weno_cell_fast<K>(x, eps, vl[i], vr[i]);
    }}
}}
extern "C" void reconstruct(int k, long n, const double *v, double eps, double *vl, double *vr)
{{
    if (k == 2) run<2>(n, v, eps, vl, vr);
    else run<3>(n, v, eps, vl, vr);
}}
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    d = tmp_path_factory.mktemp("recon")
    (d / "recon.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-mfma", "-ffp-contract=off", "-shared", "-fPIC", "-o", str(d / "recon.so"),
                    str(d / "recon.cpp")], check=True)
    lib = C.CDLL(str(d / "recon.so"))

    def run(v, k, eps):
        vl, vr = np.empty_like(v), np.empty_like(v)
        p = C.POINTER(C.c_double)
        lib.reconstruct(k, C.c_long(v.size), v.ctypes.data_as(p), C.c_double(eps), vl.ctypes.data_as(p), vr.ctypes.data_as(p))
        return vl, vr
    return run


def states(n):
    rng = np.random.default_rng(17)
    sign = rng.choice([-1.0, 1.0], n)
    yield "small", sign * 10.0 ** rng.uniform(-323, -240, n)
    yield "zeros", np.where(rng.random(n) < 0.7, 0.0, sign * 10.0 ** rng.uniform(-300, -8, n))
    yield "ordinary", sign * 10.0 ** rng.uniform(-8, 8, n)
    yield "large", sign * 10.0 ** rng.uniform(25, 34, n)
    yield "overflow", sign * 10.0 ** rng.uniform(33.5, 39, n)
    yield "sums at the overflow", sign * rng.uniform(2e38, 3.6e38, n)
    yield "they and zeros", sign * rng.uniform(2e38, 3.6e38, n) * (rng.random(n) < 0.5)
    yield "overflow of pairs", sign * 10.0 ** rng.uniform(58, 80, n)
    yield "mixed", sign * 10.0 ** rng.uniform(-320, 60, n)
    yield "flat", np.full(n, 3e37)
    s = sign * 10.0 ** rng.uniform(-2, 2, n)
    s[::40], s[7::40] = np.inf, np.nan
    yield "not finite", s


@pytest.mark.parametrize("eps", [3e-16, 1e-6, 10.0])
@pytest.mark.parametrize("k", [2, 3])
def test_range(host, hh, dev, k, eps):
    import torch
    for name, v in states(3000):
        t = torch.as_tensor(v, device=dev)
        vl, vr = hh.Weno(v.size, k, eps).reconstruct(t)
        hl, hr = host(v, k, eps)
        for got, ref in ((vl.cpu().numpy(), hl), (vr.cpu().numpy(), hr)):
            tiny = np.abs(ref) < 1e-240
            assert np.array_equal(got[~tiny], ref[~tiny], equal_nan=True), name
            assert np.all(np.abs(got[tiny] - ref[tiny]) <= 2 * np.spacing(np.abs(ref[tiny]))), name
