"""unit_turn (phase_eval.h), the sine and cosine of in-place phases, compiled for the host from
the header's own text and compared with 80-bit functions over its whole argument range: the
FP64 form gives the nearest double or its neighbour (an error of at most 1.5 units in the last
place), the FP32 form is within 2^-36."""

import os
import re
import shutil
import subprocess

import pytest

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cuda-cvdv_amd", "csrc",
                      "phase_eval.h")

MAIN = r"""
int main() {
    const long double PI = 3.14159265358979323846264338327950288L;
    unsigned long long s = 88172645463325252ull;
    long double ulps = 0, single = 0;
    auto check = [&](double f) {
        const long double n4 = rintl(4.0L * f), r = (2.0L * f - 0.5L * n4) * PI;
        const long double sn = sinl(r), cs = cosl(r);
        const int k = (int)n4 & 3;
        const long double S = k == 0 ? sn : k == 1 ? cs : k == 2 ? -sn : -cs;
        const long double C = k == 0 ? cs : k == 1 ? -sn : k == 2 ? -cs : sn;
        auto off = [](double v, long double exact) {
            const double d = fabs((double)exact);
            return d < 1e-290 ? fabsl(v - exact) : fabsl(v - exact) / (nextafter(d, 2.0) - d);
        };
        const double2 u = unit_turn(f, 0.0), w = unit_turn(f, 0.0f);
        ulps = fmaxl(ulps, fmaxl(off(u.x, C), off(u.y, S)));
        single = fmaxl(single, fmaxl(fabsl(w.x - C), fabsl(w.y - S)));
    };
    for (int i = -512; i <= 512; ++i) {  // quarter turns, eighths, and their neighbours
        const double f = i / 1024.0;
        check(f);
        if (i > -512) check(nextafter(f, -1.0));
        if (i < 512) check(nextafter(f, 1.0));
    }
    for (int i = 0; i < 400000; ++i) {
        s ^= s << 13; s ^= s >> 7; s ^= s << 17;
        const double f = (double)(s >> 11) * 0x1p-53 - 0.5;
        check(f);
        check(f * 0x1p-10);
        check(f * 0x1p-40);
    }
    printf("%.6Lf %.6Le\n", ulps, single);
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="no host compiler")
def test_unit_turn(tmp_path):
    with open(HEADER) as f:
        body = re.sub(r"^#(pragma once|include).*$", "", f.read(), flags=re.M)
    src = tmp_path / "unit_turn.cpp"
    src.write_text("#include <cmath>\n#include <cstdio>\nusing namespace std;\n#define __device__\n"
                   "#define __forceinline__ inline\nstruct double2 { double x, y; };\n"
                   "static double2 make_double2(double a, double b) { return {a, b}; }\n" + body + MAIN)
    exe = tmp_path / "unit_turn"
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-o", str(exe), str(src)], check=True)
    ulps, single = map(float, subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split())
    assert ulps <= 1.5
    assert single <= 2.0 ** -36
