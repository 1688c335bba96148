"""Fused passes of complex64 digits of 2^7 points in two stages, against the oracle: equal
digits, one of the two, high and low, one and several column groups, runs too short for it
(the tile kernel), longer digits, tables by row, affine and other generic terms.  Bars as in test_gpu_fusion.py."""

import numpy as np
import pytest

from golden_cases import apply_ops, build_sep
from oracle.cvdv_oracle import CvdvOracle
from oracle.separable_np import SeparableStateNP
from test_gpu_fusion import _bars, _chain_ops, _loss, _run

pytestmark = pytest.mark.gpu

SHAPES = [([1, 14, 5], 51, 40), ([1, 14, 7], 52, 30), ([2, 13, 6], 53, 40), ([1, 15, 5], 54, 30), ([16, 5], 55, 30),
          ([1, 16, 6], 56, 20), ([14, 2, 6], 57, 30), ([4, 14, 3], 58, 30)]


@pytest.mark.parametrize("regs,seed,n", SHAPES, ids=["x".join(map(str, s[0])) for s in SHAPES])
def test_two_stage_digits_against_oracle(regs, seed, n):
    print(f"[two-stage] {regs}", flush=True)
    init = [["setUniform", r] if q < 3 else ["setCoherent", r, [0.3 * r, -0.4]] for r, q in enumerate(regs)]
    ops = _chain_ops(np.random.default_rng(seed), regs, n)
    h = _run(regs, init, ops, "mixed")
    o = CvdvOracle(regs, convention="cuda")
    o.initStateVector(build_sep(SeparableStateNP, regs, init))
    apply_ops(o, ops)
    hs, os_ = h.getState(), o.getState()
    err = np.max(np.abs(hs - os_)) / np.max(np.abs(os_))
    fl = _loss(hs, os_)
    print(f"    rel max amp err {err:.3e}, fidelity loss {fl:.3e}", flush=True)
    ea, ef = _bars("mixed")
    assert err <= ea and fl <= ef
