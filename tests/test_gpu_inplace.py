"""Phase programs evaluated in place (states up to 2^20 amplitudes, at most four
terms) against the oracle: every term kind pending at a qubit gate, a conditional
parity and a flush, with and without controls, on both sides of the size and of the
term count where tables take over.  Bars as in test_gpu_parity.py."""

import numpy as np
import pytest

from golden_cases import apply_ops, build_sep
from oracle.cvdv_oracle import CvdvOracle
from oracle.separable_np import SeparableStateNP

pytestmark = pytest.mark.gpu

PHASES = [["sheer", 1, 0.21], ["phaseCubic", 2, 0.03], ["q1q2", 1, 2, -0.17], ["rz", 0, 0, 0.9],
          ["cd", 1, 0, 1, [0.0, 0.4]], ["cd", 2, 0, 0, [0.0, -0.3]], ["d", 2, [0.0, 0.6]]]


@pytest.mark.parametrize("prec", ["complex128", "mixed"])
@pytest.mark.parametrize("regs", [[2, 3, 4], [2, 6, 5], [2, 9, 9], [2, 10, 9]], ids=lambda r: "x".join(map(str, r)))
def test_inplace_programs(regs, prec):
    from hipcvdv import HipCvdv, SeparableState

    print(f"[inplace] {regs} {prec}", flush=True)
    init = [["setUniform", 0], ["setCoherent", 1, [0.4, 0.2]], ["setCoherent", 2, [-0.3, 0.5]]]
    h, o = HipCvdv(regs, precision=prec), CvdvOracle(regs, convention="cuda")
    h.initStateVector(build_sep(SeparableState, regs, init, device="cuda"))
    o.initStateVector(build_sep(SeparableStateNP, regs, init))
    ea, ef = (1e-11, 1e-12) if prec == "complex128" else (5e-5, 1e-6)
    for n in (1, 3, 4, 5, 7):
        for closing in (["h", 0, 0], ["ry", 0, 1, 0.4], ["cp", 1, 0, 1], ["cp", 2, 0, 0]):
            ops = PHASES[:n] + [["p", 1], closing]
            apply_ops(h, ops)
            apply_ops(o, ops)
        apply_ops(h, PHASES[7 - n:])
        apply_ops(o, PHASES[7 - n:])
        a, b = h.getState(), o.getState()  # a flush
        assert np.max(np.abs(a - b)) <= ea * np.max(np.abs(b)), n
        assert 1 - abs(np.vdot(a, b)) ** 2 / (np.vdot(a, a).real * np.vdot(b, b).real) <= ef, n
