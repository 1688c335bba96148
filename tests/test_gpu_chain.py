"""Transforms that one gate applies to a register run as one launch (a chain) where a
tile holds whole rows of the field.  Circuits of every gate kind against the oracle
(FP64, 'cuda' convention) over the shapes where the chain's tile changes: fields of 3
to 13 points bits, contiguous and strided, narrow column runs, several blocks a tile,
states below one workgroup and above the chains' largest, fields too long for a tile.
Bars as in test_gpu_parity.py: complex128 1e-11 relative amplitude error and 1e-12
fidelity loss; mixed 5e-5 and 1e-6."""

import ctypes

import numpy as np
import pytest

from golden_cases import apply_ops, build_sep
from oracle.cvdv_oracle import CvdvOracle
from oracle.separable_np import SeparableStateNP

pytestmark = pytest.mark.gpu

SHAPES = [[1, 3], [2, 4, 3], [1, 6, 5], [3, 8], [1, 10], [8, 1, 2], [2, 7, 7], [9, 1, 3], [10, 1, 2], [11, 1, 2],
          [1, 12, 3], [2, 12], [13, 1], [1, 13], [3, 5, 9], [1, 9, 9], [4, 10, 6], [3, 10, 10],
          [3, 9, 12], [4, 8, 12]]


def _ops(rng, regs, n):
    osc = [r for r, q in enumerate(regs) if q >= 3]
    ctl = [r for r, q in enumerate(regs) if q < 3] or [osc[0]]
    a, b = osc[0], osc[-1]
    ops = []
    for _ in range(n):
        t = int(rng.choice(osc))
        c = int(rng.choice([x for x in ctl if x != t] or [x for x in range(len(regs)) if x != t]))
        q = int(rng.integers(0, regs[c]))
        th, rr = float(rng.uniform(-3, 3)), float(rng.uniform(0.05, 0.3))
        al = [float(rng.uniform(-0.6, 0.6)), float(rng.uniform(-0.6, 0.6))]
        kinds = [["d", t, al], ["s", t, rr], ["s", t, -rr], ["r", t, th], ["cd", t, c, q, al], ["cr", t, c, q, th],
                 ["cs", t, c, q, rr], ["ftQ2P", t], ["ftP2Q", t], ["sheer", t, 0.1 * th], ["phaseCubic", t, 0.02],
                 ["p", t], ["cp", t, c, q], ["rx", c, q, th], ["rz", c, q, th], ["h", c, q]]
        if a != b:
            small = 0.4 * th
            kinds += [["bs", a, b, th if regs[a] == regs[b] else small], ["q1q2", a, b, 0.1 * th],
                      ["bs", b, a, small]]
            if c not in (a, b):
                kinds += [["cbs", a, b, c, q, small], ["cbs", b, a, c, q, -small]]
        ops.append(kinds[int(rng.integers(0, len(kinds)))])
    return ops


@pytest.mark.parametrize("prec", ["complex128", "mixed"])
@pytest.mark.parametrize("regs", SHAPES, ids=lambda r: "x".join(map(str, r)))
def test_chains_against_oracle(regs, prec):
    from hipcvdv import HipCvdv, SeparableState

    print(f"[chain] {regs} {prec}", flush=True)
    rng = np.random.default_rng(sum(regs) * 7 + len(regs))
    init = [["setUniform", r] if q < 3 else ["setCoherent", r, [0.4, -0.3 + 0.2 * r]] for r, q in enumerate(regs)]
    ops = _ops(rng, regs, 24 if sum(regs) > 20 else 60)
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
    ea, ef = (1e-11, 1e-12) if prec == "complex128" else (5e-5, 1e-6)
    assert err <= ea and loss <= ef


def _fft_launches(h, gate, *args):
    h._lib.cvdvProfileEnable(h.ctx, 1)
    getattr(h, gate)(*args)
    n = h._lib.cvdvProfileRead(h.ctx, 0, None, None)
    h._lib.cvdvProfileEnable(h.ctx, 0)
    return n


def test_one_launch_a_gate():
    """A squeezing gate's four transforms, a displacement's two: one launch; a beam
    splitter's four: three; whole transforms (fusion off) one each."""
    from hipcvdv import HipCvdv, SeparableState

    h = HipCvdv([1, 8, 8])
    sep = SeparableState([1, 8, 8])
    sep.setUniform(0)
    sep.setCoherent(1, 0.3)
    sep.setCoherent(2, -0.2j)
    h.initStateVector(sep)
    assert _fft_launches(h, "s", 1, 0.2) == 1
    assert _fft_launches(h, "cd", 2, 0, 0, 0.3 + 0.1j) == 1
    assert _fft_launches(h, "bs", 1, 2, 0.4) == 3
    assert _fft_launches(h, "ftQ2P", 1) == 1
    h._c("cvdvSetTransformFusion", ctypes.c_int(0))
    assert _fft_launches(h, "s", 1, 0.2) == 4
