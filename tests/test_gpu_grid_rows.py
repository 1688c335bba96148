"""The operands of the grid readouts against the oracle: register sizes below, inside
and above the row kernels' range, ragged point lists, one and several slices, and
windows whose Gaussian leaves grid points out (registers of 2^12 points and more).
Tolerance as for the other grid readouts: 1e-12 of the largest value (sums of up to
2^14 products in FP64)."""

import numpy as np
import pytest

from oracle.cvdv_oracle import CvdvOracle

pytestmark = pytest.mark.gpu


def _pair(regs, seed):
    from hipcvdv import HipCvdv

    rng = np.random.default_rng(seed)
    n = 1 << sum(regs)
    psi = rng.normal(size=n) + 1j * rng.normal(size=n)
    psi /= np.linalg.norm(psi)
    h, o = HipCvdv(regs), CvdvOracle(regs, convention="cuda")
    h.initFromArray(psi)
    o.initFromArray(psi)
    return h, o, psi


@pytest.mark.parametrize("regs,r", [([2, 1], 1), ([2, 2], 1), ([1, 3], 1), ([4, 2], 0), ([2, 5], 1), ([8], 0),
                                    ([3, 9], 1), ([10, 1], 0), ([1, 12], 1), ([1, 13], 1), ([14], 0)], ids=str)
def test_grid_operands(regs, r):
    print(f"[grid rows] {regs} {r}", flush=True)
    h, o, _ = _pair(regs, 3 * sum(regs) + r)
    xs = np.concatenate([np.linspace(-3.1, 2.7, 6), [o._x(r)[1], 0.5 * o.grid_steps[r]]])
    ps = np.linspace(-2.9, 4.0, 5)
    for per in (False, True):
        for native in (False, True):
            got = h.getWignerGrid(r, xs, ps, per_slice=per, native=native)
            exp = o.getWignerGrid(r, xs, ps, per_slice=per, native=native)
            assert np.max(np.abs(got - exp)) <= 1e-12 * np.max(np.abs(exp)), (per, native)
        got, exp = h.getHusimiQGrid(r, xs, ps, per_slice=per), o.getHusimiQGrid(r, xs, ps, per_slice=per)
        assert np.max(np.abs(got - exp)) <= 1e-12 * np.max(np.abs(exp)), per


@pytest.mark.parametrize("qs", [[0.0], [-7.0, 3.5], [60.0, 75.0], [-500.0, 1.0]], ids=str)
def test_husimi_window_leaves_points_out(qs):
    print(f"[grid rows] window {qs}", flush=True)
    h, o, _ = _pair([1, 13], 11)
    ps = np.linspace(-5.0, 5.0, 7)
    got, exp = h.getHusimiQGrid(1, qs, ps), o.getHusimiQGrid(1, qs, ps)
    assert np.max(np.abs(got - exp)) <= 1e-12 * np.max(np.abs(exp))


def test_points_left_out_still_carry_nan():
    """0 * NaN is NaN: a slice with a non-finite amplitude outside the window reads NaN,
    the other slice is untouched."""
    h, _, psi = _pair([1, 13], 12)
    clean = h.getHusimiQGrid(1, [0.0, 1.0], [0.5], per_slice=True)
    psi[5] = np.inf
    h.initFromArray(psi)
    got = h.getHusimiQGrid(1, [0.0, 1.0], [0.5], per_slice=True)
    assert np.all(np.isnan(got[0]))
    np.testing.assert_array_equal(got[1], clean[1])
