"""Reading the state out of a lazy layout (registers swapped and reflected, phases
pending) through the tiled move, against the oracle: few and many registers, fields that
swap the contiguous end, one-bit registers, states smaller than a tile; the readout
leaves the state as it was (gates after it, a second readout, a program that needs
passes of its own).  Bars as in test_gpu_parity.py."""

import numpy as np
import pytest

from oracle.cvdv_oracle import CvdvOracle

pytestmark = pytest.mark.gpu

SHAPES = [[2], [1, 1, 1], [3, 3], [1, 4, 4], [6, 6], [5, 2, 5, 5], [1] * 13, [7, 1, 7], [4, 9, 4], [9, 9], [10, 10, 1]]


@pytest.mark.parametrize("prec", ["complex128", "mixed"])
@pytest.mark.parametrize("regs", SHAPES, ids=lambda r: "x".join(map(str, r)))
def test_lazy_layouts(regs, prec):
    from hipcvdv import HipCvdv

    print(f"[state readout] {regs} {prec}", flush=True)
    rng = np.random.default_rng(sum(regs) + 31 * len(regs))
    n = 1 << sum(regs)
    psi = rng.normal(size=n) + 1j * rng.normal(size=n)
    psi /= np.linalg.norm(psi)
    h, o = HipCvdv(regs, precision=prec), CvdvOracle(regs, convention="cuda")
    h.initFromArray(psi)
    o.initFromArray(psi)
    tol = (1e-11 if prec == "complex128" else 5e-5) * np.max(np.abs(psi))

    def check():
        exp = o.getState()
        assert np.max(np.abs(h.getState() - exp)) <= tol
        assert np.max(np.abs(h.getStateTensor().cpu().numpy() - exp)) <= tol

    def both(name, *args):
        getattr(h, name)(*args)
        getattr(o, name)(*args)

    for _ in range(3):
        for _ in range(4):
            a, b = int(rng.integers(len(regs))), int(rng.integers(len(regs)))
            if regs[a] == regs[b] and a != b:
                both("swap", a, b)
            both("p", int(rng.integers(len(regs))))
        check()                        # moved and reflected
        r = int(rng.integers(len(regs)))
        both("sheer", r, 0.3)
        both("rz", r, 0, 0.7)
        check()                        # with phases pending
        both("ftQ2P", r)
        check()                        # the readouts left the state as it was
    for r in range(len(regs)):         # more terms than tables
        both("sheer", r, 0.1)
        both("phaseCubic", r, 0.02)
        for c in range(len(regs)):
            if c != r:
                both("cd", r, c, 0, 0.2j)
    check()
    both("h", 0, 0)
    check()
