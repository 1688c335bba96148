"""The FP32 constants W_32^e of the row and fused kernels (fft_radix16.h), compiled for the host
from the header's own text.  Each is within an ulp of the exact value, and the mean of |w|^2 - 1
over the constants that one input of a butterfly meets (all its outputs equally, output 0 without
one) is at most 5e-9: a state concentrated on that input grows or shrinks by it at every stage,
and a nearest rounding's 6e-8 is met by no set of eight as a whole."""

import math
import os
import shutil
import subprocess

import numpy as np
import pytest

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cuda-cvdv_amd", "csrc",
                      "fft_radix16.h")


def _constants(tmp_path, inner):
    with open(HEADER) as f:
        text = f.read()
    body = text[text.index("template <typename R, int E, bool INNER> struct W32;"):text.index("template <int E, bool INNER = false")]
    rows = "".join(f"    show<{e}>();\n" for e in range(32))
    src = tmp_path / "w32.cpp"
    src.write_text("#include <cstdio>\n" + body + "template <int E> void show() { using W = W32<float, E, " + inner + ">; "
                   'printf("%d %d %.17g %.17g\\n", W::q, W::r, (double)W::c, (double)W::s); }\n'
                   "int main() {\n" + rows + "}\n")
    exe = tmp_path / "w32"
    subprocess.run(["g++", "-std=c++17", "-O1", "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split("\n")[:32]
    return [tuple(map(float, line.split())) for line in out]


SETS = {"true": [[k * m for m in range(1, 8)] for k in (1, 2, 3)],
        "false": [list(range(1, 16)), [2, 4, 6], [6, 12, 18]]}


@pytest.mark.skipif(not shutil.which("g++"), reason="no host compiler")
@pytest.mark.parametrize("inner", ["true", "false"])
def test_w32(tmp_path, inner):
    off = np.zeros(32)
    for e, (q, r, c, s) in enumerate(_constants(tmp_path, inner)):
        assert int(q) == e >> 3 and int(r) == e & 7
        if int(r) in (0, 4):  # multiples of an eighth turn take no constants
            continue
        a = 2 * math.pi * int(r) / 32
        for v, exact in ((c, math.cos(a)), (s, math.sin(a))):
            assert abs(v - exact) <= float(np.spacing(np.float32(exact)))
        off[e] = c * c + s * s - 1.0
    for es in SETS[inner]:
        assert abs(sum(off[e] for e in es)) <= 5e-9 * (len(es) + 1), es
