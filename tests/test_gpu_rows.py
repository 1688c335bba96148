"""Contiguous complex64 rows of 2^13 and 2^14 points, one workgroup a row and a gate's
transforms in one pass, against the oracle (FP64, 'cuda' convention): one row, fewer rows than
workgroups, many; one to four transforms; phases from tables with choice and control bits, one
factor a row, generic terms of another register, none of them; programs the row kernel does not
take (a control inside the row, more terms than one pass holds); a graph's replays.  Bars as in
test_gpu_parity.py for mixed: 5e-5 relative amplitude error, 1e-6 fidelity loss."""

import ctypes

import numpy as np
import pytest

from golden_cases import apply_ops, build_sep
from oracle.cvdv_oracle import CvdvOracle
from oracle.separable_np import SeparableStateNP

pytestmark = pytest.mark.gpu


def _gates(row, other, ctl, q):
    """One program per gate kind; `row` the contiguous register, `ctl` a control outside it."""
    ops = [["d", row, [0.4, -0.3]], ["s", row, 0.2], ["r", row, 0.9], ["r", row, 2.6], ["ftQ2P", row], ["ftP2Q", row]]
    if ctl is not None:
        ops += [["h", ctl, q], ["cd", row, ctl, q, [0.3, 0.5]], ["cr", row, ctl, q, 0.6], ["cr", row, ctl, q, 1.7],
                ["cr", row, ctl, q, -1.3], ["cs", row, ctl, q, 0.15], ["rz", ctl, q, 0.8], ["cp", row, ctl, q],
                ["rx", ctl, q, 0.4], ["sheer", row, 0.05], ["phaseCubic", row, 0.002], ["s", row, -0.15]]
    if other is not None:
        ops += [["q1q2", row, other, 0.1], ["d", row, [0.2, 0.1]], ["bs", row, other, 0.5], ["bs", other, row, -0.3],
                # a control inside the row: not the row kernel's
                ["cd", other, row, 3, [0.2, 0.1]], ["s", row, 0.1], ["rz", row, 2, 0.3], ["r", row, 0.4]]
    return ops


CASES = [([14], 0, None, None, 0), ([1, 14], 1, None, 0, 0), ([3, 2, 14], 2, None, 0, 2), ([9, 14], 1, 0, None, 0),
         ([2, 6, 14], 2, 1, 0, 1), ([10, 13], 1, 0, None, 0), ([3, 7, 13], 2, 1, 0, 2), ([11, 13], 1, None, 0, 10)]


def _compare(h, o, regs):
    a, b = h.getState(), o.getState()
    err = np.max(np.abs(a - b)) / np.max(np.abs(b))
    loss = 1 - abs(np.vdot(a, b)) ** 2 / (np.vdot(a, a).real * np.vdot(b, b).real)
    print(f"    {regs} rel max amp err {err:.3e}, fidelity loss {loss:.3e}", flush=True)
    assert err <= 5e-5 and loss <= 1e-6


def _start(regs):
    from hipcvdv import HipCvdv, SeparableState

    print(f"[rows] {regs}", flush=True)
    init = [["setUniform", r] if q < 3 else ["setCoherent", r, [0.4, -0.3 + 0.2 * r]] for r, q in enumerate(regs)]
    h = HipCvdv(regs, precision="mixed")
    h.initStateVector(build_sep(SeparableState, regs, init, device="cuda"))
    o = CvdvOracle(regs, convention="cuda")
    o.initStateVector(build_sep(SeparableStateNP, regs, init))
    return h, o


@pytest.mark.parametrize("fused", [1, 0])
@pytest.mark.parametrize("regs,row,other,ctl,q", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, list) else None)
def test_rows_against_oracle(regs, row, other, ctl, q, fused):
    h, o = _start(regs)
    h._c("cvdvSetTransformFusion", ctypes.c_int(fused))
    ops = _gates(row, other, ctl, q)
    apply_ops(h, ops)
    apply_ops(o, ops)
    _compare(h, o, regs)


def test_many_controls():
    # phases under six control bits and a quadratic of its own: more than one pass's tables
    regs = [6, 3, 14]
    h, o = _start(regs)
    ops = [["cd", 2, 0, q, [0.05 * q, 0.3]] for q in range(6)]
    ops += [op for q in range(6) for op in (["cs", 2, 0, q, 0.02], ["cr", 2, 0, q, 0.1])] + [["s", 2, 0.1]]
    apply_ops(h, ops)
    apply_ops(o, ops)
    _compare(h, o, regs)


@pytest.mark.parametrize("regs", [[2, 14], [10, 13]])
def test_replays(regs):
    h, o = _start(regs)
    ops = [["s", 1, 0.1], ["cd", 1, 0, 1, [0.3, -0.2]], ["cr", 1, 0, 1, 1.8], ["cs", 1, 0, 1, 0.1]]
    with h.capture() as g:
        apply_ops(h, ops)
    for _ in range(3):
        g.launch()
        apply_ops(o, ops)
        apply_ops(h, [["d", 1, [0.1, 0.1]]])
        apply_ops(o, [["d", 1, [0.1, 0.1]]])
        h.synchronize()
        _compare(h, o, regs)


def test_one_pass_a_gate():
    h, _ = _start([1, 14])
    h._lib.cvdvProfileEnable(h.ctx, 1)
    h.s(1, 0.2)
    n = h._lib.cvdvProfileRead(h.ctx, 0, None, None)
    h._lib.cvdvProfileEnable(h.ctx, 0)
    assert n == 1
