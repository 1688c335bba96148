"""Contiguous rows of 2^12 complex128 points, one workgroup a row and a gate's transforms in one
pass (states above 2^22), and the neighbouring lengths, which keep their tiles, against the oracle
with the gates of test_gpu_rows.py.  Bars as in test_gpu_parity.py: complex128 1e-11 relative amplitude error and
1e-12 fidelity loss; mixed 5e-5 and 1e-6."""

import ctypes

import numpy as np
import pytest

from golden_cases import apply_ops, build_sep
from oracle.cvdv_oracle import CvdvOracle
from oracle.separable_np import SeparableStateNP
from test_gpu_rows import _gates

pytestmark = pytest.mark.gpu

CASES = [([11, 12], "complex128", 1, None, 0, 10), ([3, 8, 12], "complex128", 2, 1, 0, 2),
         ([11, 12], "complex128", 1, 0, None, 0), ([12, 11], "complex128", 1, 0, None, 0),
         ([2, 10, 11], "complex128", 2, 1, 0, 1), ([11, 12], "mixed", 1, 0, None, 0), ([3, 8, 12], "mixed", 2, 1, 0, 0)]


@pytest.mark.parametrize("fused", [1, 0])
@pytest.mark.parametrize("regs,prec,row,other,ctl,q", CASES,
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, list) else None)
def test_rows_against_oracle(regs, prec, row, other, ctl, q, fused):
    from hipcvdv import HipCvdv, SeparableState

    print(f"[rows] {regs} {prec} fused {fused}", flush=True)
    init = [["setUniform", r] if n < 3 else ["setCoherent", r, [0.4, -0.3 + 0.2 * r]] for r, n in enumerate(regs)]
    ops = _gates(row, other, ctl, q)
    h = HipCvdv(regs, precision=prec)
    h.initStateVector(build_sep(SeparableState, regs, init, device="cuda"))
    h._c("cvdvSetTransformFusion", ctypes.c_int(fused))
    o = CvdvOracle(regs, convention="cuda")
    o.initStateVector(build_sep(SeparableStateNP, regs, init))
    apply_ops(h, ops)
    apply_ops(o, ops)
    a, b = h.getState(), o.getState()
    err = np.max(np.abs(a - b)) / np.max(np.abs(b))
    loss = 1 - abs(np.vdot(a, b)) ** 2 / (np.vdot(a, a).real * np.vdot(b, b).real)
    print(f"    rel max amp err {err:.3e}, fidelity loss {loss:.3e}", flush=True)
    ea, ef = (1e-11, 1e-12) if prec == "complex128" else (5e-5, 1e-6)
    assert err <= ea and loss <= ef
