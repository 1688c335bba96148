"""Gates of two registers above 2^22 amplitudes, complex128, where one register's transforms
are collected for a chain but keep a half pending when one runs alone (2^8 points at a stride of
16 and more), and the other's keep halves pending or not: the phase between the transforms reads
both registers.  Against the oracle; bars as in test_gpu_parity.py (1e-11, 1e-12)."""

import pytest

from test_gpu_turned_transform import _against_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("regs", [[8, 10, 5], [10, 8, 5], [8, 8, 7], [8, 11, 4], [5, 8, 10], [1, 8, 14]], ids=str)
def test_two_registers(regs):
    a, b = [r for r, q in enumerate(regs) if q >= 8]
    c = 3 - a - b
    ops = [["h", c, 0], ["bs", a, b, 0.7], ["sheer", a, 0.1], ["bs", b, a, -0.4], ["ftQ2P", a], ["q1q2", a, b, 0.02],
           ["cbs", a, b, c, 0, 0.9], ["d", b, [0.3, -0.2]], ["ftP2Q", a], ["bs", a, b, 0.5]]
    _against_oracle(regs, "complex128", ops)
