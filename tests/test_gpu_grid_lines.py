"""Traced Wigner windows on both sides of the line between the row kernel and the batched
transforms (phase_grid.hip): slice counts around 16, windows that fill the chip with rows and
windows that do not, against the oracle.  Tolerance as in test_gpu_grid_rows.py: 1e-12."""

import numpy as np
import pytest

from oracle.cvdv_oracle import CvdvOracle
from test_gpu_native_rows import _state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("native", [False, True])
@pytest.mark.parametrize("regs,r,nx", [([4, 3], 1, 5), ([5, 3], 1, 5), ([4, 6], 1, 33), ([5, 6], 1, 33), ([6, 5], 0, 16),
                                       ([7, 7], 1, 7), ([5, 9], 1, 3), ([5, 11], 1, 127), ([5, 11], 1, 128)], ids=str)
def test_lines(regs, r, nx, native):
    from hipcvdv import HipCvdv

    print(f"[grid lines] {regs} {r} {nx} {native}", flush=True)
    psi = _state(regs, "complex128", 7 * sum(regs) + r)
    h, o = HipCvdv(regs), CvdvOracle(regs, convention="cuda")
    h.initFromArray(psi)
    o.initFromArray(psi)
    xs, ps = np.linspace(-2.9, 3.1, nx), np.array([-1.3, 0.0, 0.4, 2.2])
    kw = {"per_slice": False, "native": native}
    got, exp = h.getWignerGrid(r, xs, ps, **kw), o.getWignerGrid(r, xs, ps, **kw)
    assert np.max(np.abs(got - exp)) <= 1e-12 * np.max(np.abs(exp))
