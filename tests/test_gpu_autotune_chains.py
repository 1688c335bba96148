"""The FFT tuner on fields whose transforms run as chains (states up to 2^22): no choice of it
reaches them, so there is one plan to time for each field."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["complex128", "mixed"])
@pytest.mark.parametrize("regs", [[9, 7], [5, 8, 6]], ids=str)
def test_one_plan_a_field(regs, prec):
    from hipcvdv import HipCvdv

    h = HipCvdv(regs, precision=prec)
    psi = np.zeros(1 << sum(regs), dtype=complex)
    psi[0] = 1.0
    h.initFromArray(psi)
    info = h.autotune()
    print(f"[autotune chains] {regs} {prec}: {info}", flush=True)
    assert info["plans_timed"] <= len(regs)
