"""Phases over the whole grid in complex128: at the edge of a register a gate's quadratic and
bilinear phases are hundreds of revolutions, of which an amplitude sees the fraction.  Random
states (as much at the edge as in the middle) against the same gates in 80 bits.  The
coefficients are exact multiples of the angles, so what is left is the transforms (2.5e-16
each, up to four of them), a rounded sine and cosine and a product for each phase: 2e-15.
A phase rounded before it is reduced is 2e-14 off at 2^8 points and 7e-14 at 2^10."""

import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L, CL = np.longdouble, np.clongdouble
PI = L("3.14159265358979323846264338327950288")


def _m(n):
    return (2 * np.arange(1 << n) + 1 - (1 << n)).astype(L)


def _turn(rev):
    r = 2 * PI * (rev - np.rint(rev))
    return (np.cos(r) + 1j * np.sin(r)).astype(CL)


def _ft(s, axis, inv):
    n = int(math.log2(s.shape[axis]))
    N = L(1 << n)
    shape = [1] * s.ndim
    shape[axis] = -1
    f = _turn((N - 1) * _m(n) / (4 * N)).reshape(shape)
    g = _turn(np.array([(N - 1) * (N - 1) / (4 * N)]))[0]
    if inv:
        return np.conj(_ft(np.conj(s), axis, False))
    return g * f * np.fft.fft(f * s, axis=axis) / np.sqrt(N)


def _sheer(s, axis, t, ctl=None):  # e^{i t x^2}, the other sign where the control axis is 1
    n = int(math.log2(s.shape[axis]))
    shape = [1] * s.ndim
    shape[axis] = -1
    p = _turn(L(t) * _m(n) ** 2 / (4 * L(1 << n))).reshape(shape)
    if ctl is None:
        return s * p
    c = [1] * s.ndim
    c[ctl] = 2
    one = np.array([0, 1]).reshape(c)
    return s * np.where(one == 1, np.conj(p), p)


def _q1q2(s, t):  # axes 1 and 2 of equal sizes
    n = int(math.log2(s.shape[1]))
    return s * _turn(L(t) * np.outer(_m(n), _m(n)) / (4 * L(1 << n)))[None]


def _squeeze(s, r):
    eh, emh, sq = math.exp(0.5 * r), math.exp(-0.5 * r), math.sqrt(abs(math.exp(r) - 1.0))
    s = _sheer(_ft(s, 1, False), 1, -0.5 * eh * sq)
    s = _sheer(_ft(s, 1, True), 1, 0.5 * emh * sq)
    s = _sheer(_ft(s, 1, False), 1, 0.5 * emh * sq)
    return _sheer(_ft(s, 1, True), 1, -0.5 * eh * sq)


def _crotate(s, th):
    tq, st = math.tan(th / 2.0), math.sin(th)
    s = _sheer(s, 1, -0.5 * tq, 0)
    s = _sheer(_ft(s, 1, False), 1, -0.5 * st, 0)
    return _sheer(_ft(s, 1, True), 1, -0.5 * tq, 0)


def _split(s, th):
    cq, cp = -math.tan(0.25 * th), -math.sin(0.5 * th)
    s = _q1q2(s, cq)
    s = _q1q2(_ft(_ft(s, 1, False), 2, False), cp)
    return _q1q2(_ft(_ft(s, 1, True), 2, True), cq)


GATES = {
    "sheer": ([1, 0], lambda s: _sheer(s, 1, 0.3), lambda h: (h.sheer(1, 0.3), h._c("cvdvFlush"))),
    "squeeze": ([1, 0], lambda s: _squeeze(s, 0.2), lambda h: h.s(1, 0.2)),
    "conditional rotation": ([1, 0], lambda s: _crotate(s, 0.4), lambda h: h.cr(1, 0, 0, 0.4)),
    "beam splitter": ([1, 0, 0], lambda s: _split(s, 0.7), lambda h: h.bs(1, 2, 0.7)),
}


@pytest.mark.parametrize("n", [6, 8, 10])
@pytest.mark.parametrize("gate", ["sheer", "squeeze", "conditional rotation", "beam splitter"])
def test_edge(gate, n):
    from hipcvdv import HipCvdv

    shape, ref, go = GATES[gate]
    regs = [q or n for q in shape]
    rng = np.random.default_rng(n)
    psi = rng.normal(size=[1 << q for q in regs]) + 1j * rng.normal(size=[1 << q for q in regs])
    psi /= np.linalg.norm(psi)
    h = HipCvdv(regs)
    h.initFromArray(psi.reshape(-1))
    go(h)
    err = np.linalg.norm((h.getState().reshape(psi.shape) - ref(psi.astype(CL))).astype(np.complex128))
    print(f"[edge accuracy] {gate} {regs}: {err:.3e}", flush=True)
    assert err <= 2e-15


@pytest.mark.parametrize("regs", [[12, 12], [11, 12], [10, 13]], ids=str)
def test_rows_under_a_bilinear_phase(regs):
    """A transform of contiguous rows above 2^22 amplitudes with e^{i t q1 q2} pending: the term is
    affine in the row, its slope up to a quarter revolution a point.  Rows of the edge and the
    middle by themselves; relative to each row.  (Unequal sizes round the coefficient itself, by
    2^-53 of up to 2^8 revolutions, so they are compared with the coefficient that is held.)"""
    import torch
    from hipcvdv import HipCvdv

    a, n = regs
    t = 0.7
    g = torch.Generator(device="cuda").manual_seed(9)
    psi = torch.view_as_complex(torch.randn(1 << a, 1 << n, 2, dtype=torch.float64, device="cuda", generator=g))
    psi /= torch.linalg.vector_norm(psi)
    h = HipCvdv(regs)
    h.initFromArray(psi.reshape(-1))
    h.q1q2(0, 1, t)
    h.ftQ2P(1)
    rows = [0, 1, (1 << a - 1) - 1, (1 << a) - 2, (1 << a) - 1]
    got = h.getStateTensor().reshape(psi.shape)[rows].cpu().numpy()
    src = psi[rows].cpu().numpy().astype(CL)
    c = t / (4.0 * 2 ** n) if a == n else t * h.grid_steps[0] * h.grid_steps[1] / (8.0 * math.pi)
    exp = _ft(src * _turn(L(c) * np.outer(_m(a)[rows], _m(n))), 1, False)
    err = np.linalg.norm((got - exp).astype(complex), axis=1) / np.linalg.norm(exp.astype(complex), axis=1)
    print(f"[edge accuracy] rows {regs}: {err}", flush=True)
    assert np.max(err) <= 1e-15
