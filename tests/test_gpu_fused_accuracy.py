"""The error of fused passes in mixed precision is no larger than that of the same transforms
run as half passes of the tile kernel.  Four centred Fourier transforms are the identity, so
the state after 4 k of them is the one they started from, and the distance from it is their
error alone.  Eight transforms; digits of 2^7 points in two stages ([14,5], [14,6]) and in the
tile kernel ([12,6] and [16,5], digits of 2^6 and 2^8).  The relative difference between two
such errors over 2^18 amplitudes and more has a spread of 2^-10 (independent roundings), which
is the margin."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("regs", [[14, 5], [14, 6], [12, 6], [16, 5]], ids=str)
def test_fused_error(regs):
    from hipcvdv import HipCvdv

    rng = np.random.default_rng(sum(regs))
    n = 1 << sum(regs)
    psi = rng.normal(size=n) + 1j * rng.normal(size=n)
    psi = (psi / np.linalg.norm(psi)).astype(np.complex64).astype(np.complex128)
    err = []
    for fuse in (0, 1):
        h = HipCvdv(regs, precision="mixed")
        h._c("cvdvSetTransformFusion", ctypes.c_int(fuse))
        h.initFromArray(psi)
        for _ in range(8):
            h.ftQ2P(0)
        err.append(np.linalg.norm(h.getState() - psi))
    print(f"[fused accuracy] {regs}: half passes {err[0]:.4e}, fused {err[1]:.4e}", flush=True)
    assert err[1] <= err[0] * (1 + 2 ** -10)
