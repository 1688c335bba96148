"""Conditional quarter turns (a transform whose direction the control bit chooses) against
the oracle (FP64, 'cuda' convention), with pending phases and stored reflections, at the
shapes where the route changes: control above the field, among a tile's columns, among its
blocks, inside the field's neighbour, in a register that is itself transformed; chains, one
pass, rows of 2^13 and 2^14 points, the four-step split.  Bars as in test_gpu_parity.py:
complex128 1e-11 relative amplitude error (1e-10 above 2^13 points) and 1e-12 fidelity
loss; mixed 5e-5 and 1e-6."""

import math

import numpy as np
import pytest

from golden_cases import apply_ops, build_sep
from oracle.cvdv_oracle import CvdvOracle
from oracle.separable_np import SeparableStateNP

pytestmark = pytest.mark.gpu

ROTATIONS = [
    ([1, 3], 1, 0, 0), ([6, 1], 0, 1, 0), ([2, 6], 1, 0, 1), ([3, 5, 4], 1, 2, 0), ([3, 5, 4], 1, 2, 3),
    ([4, 10, 6], 1, 0, 3), ([1, 12], 1, 0, 0), ([12, 2], 0, 1, 1), ([9, 13], 1, 0, 8), ([10, 13], 1, 0, 0),
    ([9, 14], 1, 0, 8), ([13, 10], 0, 1, 2), ([11, 12], 1, 0, 10), ([12, 11], 0, 1, 0), ([12, 8, 3], 1, 0, 11),
]
SPLITTERS = [([1, 6, 6], 1, 2, 0, 0), ([6, 2, 6], 2, 0, 1, 1), ([1, 11, 11], 1, 2, 0, 0),
             ([6, 6], 0, 1, 1, 2), ([6, 6], 0, 1, 0, 5)]


def _against_oracle(regs, prec, ops):
    from hipcvdv import HipCvdv, SeparableState

    print(f"[turned] {regs} {prec} {ops[-1]}", flush=True)
    init = [["setUniform", r] if q < 3 else ["setCoherent", r, [0.4, -0.3 + 0.2 * r]] for r, q in enumerate(regs)]
    h = HipCvdv(regs, precision=prec)
    h.initStateVector(build_sep(SeparableState, regs, init, device="cuda"))
    o = CvdvOracle(regs, convention="cuda")
    o.initStateVector(build_sep(SeparableStateNP, regs, init))
    apply_ops(h, ops)
    apply_ops(o, ops)
    a, b = h.getState(), o.getState()
    err = np.max(np.abs(a - b)) / np.max(np.abs(b))
    loss = 1 - abs(np.vdot(a, b)) ** 2 / (np.vdot(a, a).real * np.vdot(b, b).real)
    print(f"    rel max amp err {err:.3e}, fidelity loss {loss:.3e}", flush=True)
    ea, ef = (1e-11 if max(regs) <= 13 else 1e-10, 1e-12) if prec == "complex128" else (5e-5, 1e-6)
    assert err <= ea and loss <= ef


@pytest.mark.parametrize("prec", ["complex128", "mixed"])
@pytest.mark.parametrize("regs,tgt,creg,cq", ROTATIONS)
def test_conditional_rotation(regs, tgt, creg, cq, prec):
    quarter = math.pi / 2
    ops = []
    for turn, reflect in ((1, None), (-1, creg), (1, tgt), (-1, None), (3, creg)):
        if reflect is not None:
            ops.append(["p", reflect])
        ops += [["sheer", tgt, 0.05], ["rz", creg, cq, 0.4], ["cr", tgt, creg, cq, turn * quarter + 0.3],
                ["rx", creg, cq, 0.7]]
    ops.append(["cr", tgt, creg, cq, quarter])
    _against_oracle(regs, prec, ops)


@pytest.mark.parametrize("prec", ["complex128", "mixed"])
@pytest.mark.parametrize("regs,r1,r2,creg,cq", SPLITTERS)
def test_conditional_beam_splitter(regs, r1, r2, creg, cq, prec):
    ops = [["rx", creg, cq, 0.5], ["cbs", r1, r2, creg, cq, math.pi + 0.4], ["rx", creg, cq, 0.5],
           ["cbs", r1, r2, creg, cq, 3 * math.pi - 0.2]]
    _against_oracle(regs, prec, ops)
