"""cvdvGetStateDevice into the destinations that it takes: a tensor of its own, and a buffer
aligned to its doubles only (complex128: a kernel of 16-byte stores, or a plain copy), with
nothing pending, with phases pending and with registers moved.  The same values bit for bit
in both (the same arithmetic), and cvdvGetState's."""

import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["complex128", "mixed"])
@pytest.mark.parametrize("regs", [[2], [3, 3], [1, 5, 5], [9, 9]], ids=str)
def test_destinations(regs, prec):
    from hipcvdv import HipCvdv

    print(f"[state tensor] {regs} {prec}", flush=True)
    rng = np.random.default_rng(sum(regs))
    n = 1 << sum(regs)
    psi = rng.normal(size=n) + 1j * rng.normal(size=n)
    h = HipCvdv(regs, precision=prec)
    h.initFromArray(psi / np.linalg.norm(psi))
    for step in range(3):
        if step:
            h.sheer(0, 0.2)
        if step == 2:
            h.p(len(regs) - 1)
            if len(regs) > 1:
                h.swap(len(regs) - 2, len(regs) - 1)
        own = h.getStateTensor()
        raw = torch.zeros(2 * n + 2, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()  # filled on torch's stream, written on the simulator's
        if prec == "complex128":
            h._c("cvdvGetStateDevice", ctypes.c_void_p(raw.data_ptr() + 8))
            torch.testing.assert_close(raw[1:-1], torch.view_as_real(own).reshape(-1), rtol=0, atol=0)
            assert raw[0] == 0 and raw[-1] == 0
        np.testing.assert_array_equal(h.getState(), own.cpu().numpy())
