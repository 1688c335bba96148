"""Conditional quarter turns (a transform whose direction the control bit chooses) under many
pending conditional phases: more terms than one launch of such a transform holds, with the
turning control's own phase among them (the transform's linear term then shares its slot) and
without it.  Strided fields that only chains serve at these sizes, and contiguous ones whose
one-pass tile spans the control bit.  Against the oracle (FP64, 'cuda' convention); bars as in
test_gpu_parity.py: complex128 1e-11 relative amplitude error and 1e-12 fidelity loss; mixed
5e-5 and 1e-6."""

import math

import pytest

from test_gpu_turned_transform import _against_oracle

pytestmark = pytest.mark.gpu

QUARTER = math.pi / 2


def _controls(regs, tgt):
    """(register, qubit) of every bit outside the target, the target's neighbours first."""
    out = [(r, q) for r in range(len(regs)) if r != tgt for q in range(regs[r])]
    return sorted(out, key=lambda c: (abs(c[0] - tgt), -c[1] if c[0] < tgt else c[1]))


# (registers, target): strided by 2^8, 2^10, 2^7; contiguous under single qubits (the control
# next to the field) and under one register
SHAPES = [([10, 8], 0), ([9, 10], 0), ([10, 7], 0), ([1] * 8 + [8], 8), ([1] * 7 + [9], 7), ([8, 9], 1),
          ([10] + [1] * 8, 0), ([6, 12], 0)]


@pytest.mark.parametrize("prec", ["complex128", "mixed"])
@pytest.mark.parametrize("turn", [1, -1])
@pytest.mark.parametrize("count", [6, 7, 8, 12])
@pytest.mark.parametrize("regs,tgt", SHAPES)
def test_conditional_rotation(regs, tgt, count, turn, prec):
    ctl = _controls(regs, tgt)
    many = ctl[:count]
    ops = []
    for creg, cq in (many[0], many[-1]):
        ops += [["cd", tgt, r, q, [0.0, 0.3 - 0.02 * i]] for i, (r, q) in enumerate(many)]
        ops.append(["cr", tgt, creg, cq, turn * QUARTER])
    # again, the turning control's own phase not among the pending ones
    ops += [["cd", tgt, r, q, [0.0, 0.1]] for r, q in many[:-1]]
    ops.append(["cr", tgt, creg, cq, turn * QUARTER])
    _against_oracle(regs, prec, ops)


@pytest.mark.parametrize("prec", ["complex128", "mixed"])
@pytest.mark.parametrize("count", [6, 7, 8])
@pytest.mark.parametrize("regs,r1,r2,creg", [([6, 8, 6], 0, 2, 1), ([8, 5, 5], 1, 2, 0)])
def test_conditional_beam_splitter(regs, r1, r2, creg, count, prec):
    n = min(count, regs[creg])
    ops = [["cd", r, creg, q, [0.0, 0.2]] for r in (r1, r2) for q in range(n)]
    ops.append(["cbs", r1, r2, creg, n - 1, math.pi])
    _against_oracle(regs, prec, ops)
