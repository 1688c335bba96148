"""The phase tables of a chain of rows: as much memory as its programs take, and chains whose
tables together exceed what one program may ask for (ten controls pending before a conditional
squeezing of a 2^14 row) run step by step, eagerly and in a captured graph, which reserves no
more.  Amplitudes against the oracle under the bars of test_gpu_parity.py (mixed 5e-5)."""

import numpy as np
import pytest
import torch

from golden_cases import apply_ops
from oracle.cvdv_oracle import CvdvOracle

pytestmark = pytest.mark.gpu


def test_arena_holds_the_programs_tables():
    """[11,12] complex128: the four tables of a squeezing take 256 KiB, the largest programs of
    four steps would take 24 MiB."""
    from hipcvdv import HipCvdv

    h = HipCvdv([11, 12])
    psi = torch.zeros(1 << 23, dtype=torch.complex128, device="cuda")
    psi[0] = 1.0
    h.initFromArray(psi)
    h.ftQ2P(1)
    h._c("cvdvSynchronize")
    free = torch.cuda.mem_get_info()[0]
    h.s(1, 0.2)
    h._c("cvdvSynchronize")
    used = free - torch.cuda.mem_get_info()[0]
    print(f"[row arena] {used >> 10} KiB", flush=True)
    assert used < 8 << 20


@pytest.mark.parametrize("captured", [False, True])
def test_chain_beyond_the_arena_bound(captured):
    from hipcvdv import HipCvdv

    regs, t = [1] * 10 + [14], 10
    rng = np.random.default_rng(5)
    n = 1 << sum(regs)
    x = np.arange(1 << 14) - (1 << 13)
    psi = (rng.normal(size=n) + 1j * rng.normal(size=n)) * np.tile(np.exp(-(x / 600.0) ** 2), 1 << 10)
    psi = (psi / np.linalg.norm(psi)).astype(np.complex64).astype(np.complex128)
    ops = [["cd", t, c, 0, [0.0, 0.2 + 0.01 * c]] for c in range(10)] + [["cs", t, 3, 0, 0.2]]
    h, o = HipCvdv(regs, precision="mixed"), CvdvOracle(regs, convention="cuda")
    o.initFromArray(psi)
    apply_ops(o, ops)
    exp, graph = o.getState(), None
    if captured:
        h.initFromArray(psi)
        with h.capture() as graph:
            apply_ops(h, ops)
    for _ in range(3):
        h.initFromArray(psi)
        if captured:
            graph.launch()
        else:
            apply_ops(h, ops)
        assert np.max(np.abs(h.getState() - exp)) <= 5e-5 * np.max(np.abs(exp))
