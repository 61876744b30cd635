"""The shared pieces of the EXACT reconstruction (tri3_exact, pair2_exact: formed once, used by three and
two cells) against the cell-by-cell form, compiled for the host: the same numbers for every state, also
where products overflow."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MATH = os.path.join(REPO, "hr-weno_amd", "csrc", "weno_math.hpp")

PROGRAM = f"""
#include <cmath>
#include <cstdio>
#include <random>
#include "{MATH}"
using namespace hrw;
static bool same(double a, double b) {{ return a == b || (std::isnan(a) && std::isnan(b)); }}
int main()
{{
    std::mt19937_64 g(7);
    const double big[] = {{0.0, 1e-320, 1e-160, 1e-3, 1.0, 1e30, 1e100, 1e153, 2e154, 4.4e307, 5e307, 5.9e307, 6.1e307, 8.9e307,
                          9.1e307, 1.2e308, 1.7e308, INFINITY, NAN}};
    const int nbig = sizeof big / sizeof *big;
    long wrong = 0;
    auto check = [&](const double *x) {{
        double vl, vr, wl, wr;
        weno_cell_exact<3>(x, 1e-6, nullptr, vl, vr);
        recon3_exact(1e-6, tri3_exact(x[0], x[1], x[2]), tri3_exact(x[1], x[2], x[3]), tri3_exact(x[2], x[3], x[4]), wl, wr);
        if ((!same(vl, wl) || !same(vr, wr)) && wrong++ < 3) std::printf("3: %g %g %g %g %g: %a %a, %a %a\\n", x[0], x[1], x[2], x[3], x[4], vl, vr, wl, wr);
        weno_cell_exact<2>(x, 1e-6, nullptr, vl, vr);
        recon2_exact(1e-6, pair2_exact(x[0], x[1]), pair2_exact(x[1], x[2]), wl, wr);
        if ((!same(vl, wl) || !same(vr, wr)) && wrong++ < 3) std::printf("2: %g %g %g: %a %a, %a %a\\n", x[0], x[1], x[2], vl, vr, wl, wr);
    }};
    for (int i = 0; i < 400000; ++i) {{
        double x[5];
        const int kind = (int)(g() % 4);
        const double base = big[g() % nbig];
        for (double &c : x) {{
            const double r = (double)(g() >> 11) * 0x1p-53;
            c = kind == 0 ? base : kind == 1 ? base * (1.0 + 1e-3 * (r - 0.5)) : kind == 2 ? big[g() % nbig] * (0.5 + 0.5 * r)
                                                                                 : std::exp2(2000.0 * (r - 0.5));
            if (kind >= 2 && (g() & 1)) c = -c;
        }}
        check(x);
    }}
    std::printf("%ld\\n", wrong);
}}
"""


def test_shared_pieces(tmp_path):
    src, exe = tmp_path / "pieces.cpp", tmp_path / "pieces"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split("\n")
    assert out[-2] == "0", out
