"""A non-finite amplitude in the native Wigner picture: the rows whose products read it are NaN
throughout, every other row is finite and what it was, though two rows share a transform and
from 2^7 points on neighbouring lanes share their loads (the products of lanes outside the grid
are formed and dropped).  Bound 1e-12 of the largest value, as in test_gpu_native_rows.py: the
partner row is transformed with other numbers beside it."""

import numpy as np
import pytest

from test_gpu_native_rows import _state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("regs", [[6], [7], [9], [2, 7]], ids=str)
def test_only_rows_that_read_it(regs, value):
    from hipcvdv import HipCvdv

    r = len(regs) - 1
    N = 1 << regs[r]
    psi = _state(regs, "complex128", 3)
    h = HipCvdv(regs)
    h.initFromArray(psi)
    clean = h.getWigner(r)
    for t in (0, 5, 31, 32, 63, N // 2 + 1, N - 65 if N > 65 else 1, N - 6, N - 1):
        print(f"[native non-finite] {regs} {value} {t}", flush=True)
        bad = psi.copy()
        bad[t] = value
        h.initFromArray(bad)
        got = h.getWigner(r)
        i = np.arange(N)
        hit = np.abs(t - i) <= np.minimum(i, N - 1 - i)
        assert np.all(np.isnan(got[:, hit]))
        assert np.max(np.abs(got[:, ~hit] - clean[:, ~hit])) <= 1e-12 * np.max(np.abs(clean))
