"""Husimi windows on both sides of the line between the real and the complex products
(phase_grid.hip): registers of up to 2^6 points under few and many slices, large windows and small, traced and
per slice, against the oracle (which takes every 25th column of a large window).  Tolerance as in test_gpu_grid_rows.py: 1e-12 of the largest value."""

import numpy as np
import pytest

from oracle.cvdv_oracle import CvdvOracle
from test_gpu_native_rows import _state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("regs,r,nq,np_", [([8, 1], 1, 64, 64), ([9, 1], 1, 64, 64), ([9, 2], 1, 31, 33), ([9, 3], 1, 32, 32),
                                           ([8, 4], 1, 128, 128), ([9, 4], 1, 128, 128), ([9, 4], 1, 7, 3),
                                           ([5, 9], 0, 129, 127), ([4, 10], 0, 200, 90), ([9, 5], 1, 150, 120),
                                           ([9, 6], 1, 128, 128)], ids=str)
def test_lines(regs, r, nq, np_):
    from hipcvdv import HipCvdv

    print(f"[husimi grid lines] {regs} {r} {nq} x {np_}", flush=True)
    psi = _state(regs, "complex128", 11 * sum(regs) + r)
    h, o = HipCvdv(regs), CvdvOracle(regs, convention="cuda")
    h.initFromArray(psi)
    o.initFromArray(psi)
    qs, ps = np.linspace(-2.9, 3.1, nq), np.linspace(-1.3, 2.2, np_)
    cols = slice(None, None, 25) if nq > 25 else slice(None)
    for per in (False, True):
        got, exp = h.getHusimiQGrid(r, qs, ps, per_slice=per), o.getHusimiQGrid(r, qs[cols], ps, per_slice=per)
        assert np.max(np.abs(got[..., cols] - exp)) <= 1e-12 * np.max(np.abs(exp)), per
