"""Native Wigner and Husimi readouts on both sides of the lines between the row kernels and the
routes for many slices (phase_space.hip), contiguous and strided fields, both precisions (a
mixed Wigner of 16 slices or more widens them first), against the oracle.  Tolerance as in
test_gpu_native_rows.py: N-point transforms of sums of S products in FP64, 1e-12 of the largest
value."""

import numpy as np
import pytest

from oracle.cvdv_oracle import CvdvOracle
from test_gpu_native_rows import _state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["complex128", "mixed"])
@pytest.mark.parametrize("regs,r", [([4, 4], 1), ([3, 5], 1), ([4, 5], 1), ([3, 6], 1), ([4, 6], 1), ([5, 6], 1), ([6, 3], 0),
                                    ([6, 4], 0), ([4, 7], 1), ([5, 7], 1), ([7, 3], 0), ([7, 4], 0), ([4, 8], 1),
                                    ([5, 8], 1), ([6, 8], 1), ([8, 5], 0), ([8, 6], 0), ([7, 9], 1), ([4, 10], 1)],
                         ids=str)
def test_lines(regs, r, prec):
    from hipcvdv import HipCvdv

    print(f"[native lines] {regs} {r} {prec}", flush=True)
    psi = _state(regs, prec, 5 * sum(regs) + r)
    h, o = HipCvdv(regs, precision=prec), CvdvOracle(regs, convention="cuda")
    h.initFromArray(psi)
    o.initFromArray(psi)
    for name in ("getWigner", "getHusimiQ"):
        got, exp = getattr(h, name)(r), getattr(o, name)(r)
        assert np.max(np.abs(got - exp)) <= 1e-12 * np.max(np.abs(exp)), name
