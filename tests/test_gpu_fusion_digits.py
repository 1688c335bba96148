"""Half transforms kept pending when the four-step digits differ (registers of an odd
number of qubits): circuits that chain the register's transforms against the oracle,
and the launch count.  Shapes: digits (5, 6) and (6, 7) with narrow and wide column
runs, (7, 8) contiguous with per-column twiddles, (4, 5) of a 2^9 register.
Bars as in test_gpu_fusion.py."""

import ctypes

import numpy as np
import pytest

from golden_cases import apply_ops, build_sep
from oracle.cvdv_oracle import CvdvOracle
from oracle.separable_np import SeparableStateNP
from test_gpu_fusion import PRECS, _bars, _chain_ops, _loss, _run

pytestmark = pytest.mark.gpu

SHAPES = [([1, 11, 4], 41, 50), ([2, 13, 3], 42, 50), ([1, 13, 6], 43, 40), ([1, 15], 44, 50), ([1, 9, 13], 45, 20)]


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("regs,seed,n", SHAPES, ids=["x".join(map(str, s[0])) for s in SHAPES])
def test_unequal_digits_against_oracle(regs, seed, n, prec):
    print(f"[fusion] unequal digits {regs} {prec}", flush=True)
    init = [["setUniform", 0]] + [["setCoherent", r, [0.3 * r, -0.4]] for r in range(1, len(regs))]
    ops = _chain_ops(np.random.default_rng(seed), regs, n)
    h = _run(regs, init, ops, prec)
    o = CvdvOracle(regs, convention="cuda")
    o.initStateVector(build_sep(SeparableStateNP, regs, init))
    apply_ops(o, ops)
    hs, os_ = h.getState(), o.getState()
    err = np.max(np.abs(hs - os_)) / np.max(np.abs(os_))
    fl = _loss(hs, os_)
    print(f"    rel max amp err {err:.3e}, fidelity loss {fl:.3e}", flush=True)
    ea, ef = _bars(prec)
    assert err <= ea and fl <= ef


@pytest.mark.parametrize("prec", PRECS)
def test_launch_counts(prec):
    """m transforms of a 2^13 register at stride 2^6: m + 1 launches."""
    h = _run([1, 13, 6], [["setUniform", 0], ["setCoherent", 1, 0.3], ["setCoherent", 2, 0.1]], [], prec)
    h._lib.cvdvProfileEnable(h.ctx, 1)
    for i in range(5):
        (h.ftQ2P if i % 2 == 0 else h.ftP2Q)(1)
        h.sheer(1, 0.05)
    h.flush()
    n = h._lib.cvdvProfileRead(h.ctx, 0, ctypes.byref(ctypes.c_double(0)), None)
    assert n == 6
