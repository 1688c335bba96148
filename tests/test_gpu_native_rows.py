"""The row kernels of the native Wigner and Husimi readouts (one workgroup per row
or pair of rows) against the oracle, over the register sizes where their tiles
change (several rows a workgroup below 2^9 points, a 64 KiB tile at 2^12), with
contiguous and strided fields, reflected registers, both precisions and slice
counts on both sides of the tiled sum (at most N/16 slices go by rows).  Both sides read the same amplitudes
(rounded once to complex64 in the mixed mode) in FP64.  Tolerance: N-point
transforms of rows whose entries sum S products, 2^-53 times a few hundred
roundings, relative to the largest value: 1e-12."""

import numpy as np
import pytest

from oracle.cvdv_oracle import CvdvOracle

pytestmark = pytest.mark.gpu


def _state(regs, prec, seed):
    rng = np.random.default_rng(seed)
    n = 1 << sum(regs)
    psi = rng.normal(size=n) + 1j * rng.normal(size=n)
    psi /= np.linalg.norm(psi)
    return psi.astype(np.complex64).astype(np.complex128) if prec == "mixed" else psi


@pytest.mark.parametrize("prec", ["complex128", "mixed"])
@pytest.mark.parametrize("regs,r", [([2], 0), ([3], 0), ([1, 4], 1), ([5, 1], 0), ([2, 6], 1), ([8], 0), ([1, 9], 1),
                                    ([10, 1], 0), ([1, 11], 1), ([2, 2, 6], 2), ([6, 7], 1), ([7, 6], 1), ([3, 5, 2], 1)],
                         ids=str)
def test_native_rows(regs, r, prec):
    from hipcvdv import HipCvdv

    print(f"[native rows] {regs} {r} {prec}", flush=True)
    psi = _state(regs, prec, sum(regs) + r)
    h, o = HipCvdv(regs, precision=prec), CvdvOracle(regs, convention="cuda")
    h.initFromArray(psi)
    o.initFromArray(psi)
    for reflected in (False, True):
        if reflected:
            h.p(r)
            o.p(r)
        for name in ("getWigner", "getHusimiQ", "getHusimiQWigner"):
            got, exp = getattr(h, name)(r), getattr(o, name)(r)
            assert np.max(np.abs(got - exp)) <= 1e-12 * np.max(np.abs(exp)), (name, reflected)


def test_non_finite_row_leaves_its_partner_alone():
    """A single NaN amplitude of the last point reaches only the rows whose products
    read it (here the last row alone); the row that shares its transform stays."""
    from hipcvdv import HipCvdv

    N = 64
    psi = _state([6], "complex128", 3)
    h = HipCvdv([6])
    h.initFromArray(psi)
    clean = h.getWigner(0)
    psi[N - 1] = np.nan
    h.initFromArray(psi)
    got = h.getWigner(0)
    hit = [i for i in range(N) if N - 1 - i <= min(i, N - 1 - i)]
    keep = [i for i in range(N) if i not in hit]
    assert np.all(np.isnan(got[:, hit]))
    np.testing.assert_array_equal(got[:, keep], clean[:, keep])
