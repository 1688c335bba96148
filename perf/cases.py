"""Performance cases of the simulator: what a user's program runs, and how large.

listed() holds named cases, draw() makes more of the same ranges.  prepare()
builds what a program has in hand before the call (a simulator, its initial
wavefunctions, its circuit; a loaded state for the readouts; a recorded and
tuned batch), run() is one pass through the public entry points, work() the
bytes and operations it cannot do without, exact() the same result in 64 bits by
plain torch and numpy.

A mixed-precision simulator holds complex64 amplitudes, so a program that keeps
its results keeps them at that width: run() returns them as complex64/float32.
"""

import cmath
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cuda-cvdv_amd"))

from hipcvdv import HipCvdv, HipCvdvBatch, SeparableState  # noqa: E402

PI = math.pi


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest program: one qubit and one oscillator of 2^10 points, five
        # gates and a qubit measurement; launches and calls are its whole time
        {"name": "small_circuit", "kind": "circuit", "mix": "small", "regs": "1,10", "prec": "complex128",
         "gates": 5, "graph": False},
        # every gate of the interface once, on one qubit and two oscillators of
        # 2^10 points (2^21 amplitudes): the size of the per-gate timings of the API
        {"name": "api_gates", "kind": "circuit", "mix": "api", "regs": "1,10,10", "prec": "complex128",
         "gates": 22, "graph": False},
        # Gaussian optics on two modes at 2^28 amplitudes, mixed precision: the
        # largest ordinary state
        {"name": "gaussian_large", "kind": "circuit", "mix": "gaussian", "regs": "14,14", "prec": "mixed",
         "gates": 12, "graph": False},
        # the same in full double precision, two registers of unequal size
        {"name": "gaussian_double", "kind": "circuit", "mix": "gaussian", "regs": "13,12", "prec": "complex128",
         "gates": 12, "graph": False},
        # oscillator-to-qubit state transfer, 14 qubits and 2^14 points (2^28), read
        # out as the joint qubit distribution and the state
        {"name": "transfer_large", "kind": "circuit", "mix": "transfer", "regs": ",".join(["1"] * 14 + ["14"]),
         "prec": "mixed", "gates": 42, "graph": False},
        # the same protocol at the size of a study: 4 qubits and 2^12 points
        {"name": "transfer_small", "kind": "circuit", "mix": "transfer", "regs": "1,1,1,1,12",
         "prec": "complex128", "gates": 12, "graph": False},
        # a parameter sweep: a thousand independent circuits of uneven size in one launch
        {"name": "batch_sweep", "kind": "batch", "circuits": 1024, "prec": "mixed"},
        # both phase-space pictures of one oscillator, for a figure
        {"name": "phase_small", "kind": "native", "regs": "1,10", "prec": "complex128", "wigner": True,
         "husimi": True},
        # the native Wigner grid of a 2^12-point oscillator entangled with 4 qubits
        {"name": "wigner_native", "kind": "native", "regs": "2,2,12", "prec": "complex128", "wigner": True,
         "husimi": False},
        # and its Husimi function
        {"name": "husimi_native", "kind": "native", "regs": "2,2,12", "prec": "complex128", "wigner": False,
         "husimi": True},
        # both on a 512 x 512 window, one picture for each of the 16 qubit branches
        {"name": "grid_branches", "kind": "grid", "regs": "2,2,12", "prec": "complex128", "points": 512,
         "branches": True, "native": True},
        # everything that is read off a 2^21 state without changing it: norm,
        # marginals, joint distributions, overlaps, photon numbers
        {"name": "readouts", "kind": "readouts", "regs": "1,10,10", "prec": "complex128"},
    ]


def draw(rng):
    prec = rng.choice(["complex128", "mixed"])
    kind = rng.choice(["circuit", "circuit", "circuit", "batch", "native", "grid", "readouts"])
    if kind == "circuit":
        mix = rng.choice(["small", "api", "gaussian", "transfer"])
        top = 26 if prec == "mixed" else 25
        if mix == "small":
            regs, gates = [rng.randint(1, 3), rng.randint(6, 13)], rng.randint(3, 15)
        elif mix == "api":
            regs, gates = [rng.randint(1, 2), rng.randint(5, 12), rng.randint(5, 11)], 22
        elif mix == "gaussian":
            a = rng.randint(6, 14)
            regs, gates = [a, rng.randint(6, min(14, top - a))], rng.randint(4, 12)
        else:
            osc = rng.randint(8, 14)
            q = rng.randint(2, min(12, top - osc))
            regs, gates = [1] * q + [osc], 3 * q
        graph = mix == "small" and rng.random() < 0.4
        return {"kind": kind, "mix": mix, "regs": ",".join(map(str, regs)), "prec": prec, "gates": gates,
                "graph": graph}
    if kind == "batch":
        return {"kind": kind, "circuits": int(round(2 ** rng.uniform(4.0, 9.5))), "prec": prec}
    if kind == "native":
        regs = [rng.randint(1, 4), rng.randint(6, 12)]
        if rng.random() < 0.3:  # the oscillator is not always the last register
            regs.reverse()
        w = rng.random() < 0.6
        return {"kind": kind, "regs": ",".join(map(str, regs)), "prec": prec, "wigner": w,
                "husimi": not w or rng.random() < 0.5}
    if kind == "grid":
        regs = [rng.randint(1, 4), rng.randint(7, 12)]
        return {"kind": kind, "regs": ",".join(map(str, regs)), "prec": prec,
                "points": int(round(2 ** rng.uniform(5.0, 9.0))), "branches": rng.random() < 0.6,
                "native": rng.random() < 0.5}
    regs = [rng.randint(1, 3), rng.randint(5, 12), rng.randint(4, 10)]
    return {"kind": kind, "regs": ",".join(map(str, regs)), "prec": prec}


# ---------------------------------------------------------------- circuits
def _regs(case):
    return [int(v) for v in case["regs"].split(",")]


def _disc(rng, radius):
    return cmath.rect(radius * math.sqrt(rng.random()), rng.uniform(0, 2 * PI))


def _oscillators(regs):
    return [r for r, n in enumerate(regs) if n >= 4]


def _ops(case, seed):
    """The gates (method, arguments): which ones depends on the case alone, their
    parameters on the seed."""
    regs, rng = _regs(case), random.Random(1000003 * seed + 17)
    osc = _oscillators(regs)
    if case["mix"] == "small":
        turn = [lambda: ("h", 0, 0), lambda: ("cd", 1, 0, 0, _disc(rng, 1.0)),
                lambda: ("r", 1, rng.uniform(-0.75, 0.75)), lambda: ("s", 1, rng.uniform(0.05, 0.3)),
                lambda: ("h", 0, 0), lambda: ("d", 1, _disc(rng, 1.0)), lambda: ("rx", 0, 0, rng.uniform(-PI, PI)),
                lambda: ("cr", 1, 0, 0, rng.uniform(-0.75, 0.75))]
        return [turn[i % len(turn)]() for i in range(case["gates"])]
    if case["mix"] == "gaussian":
        a, b = osc
        half = regs[a] == regs[b]  # a half turn swaps the modes: equal sizes only

        def theta():
            return rng.uniform(-PI, PI) if half else rng.uniform(-1.4, 1.4)

        turn = [lambda: ("d", a, _disc(rng, 1.0)), lambda: ("r", b, rng.uniform(-PI, PI)),
                lambda: ("bs", a, b, PI / 2 if half else 1.2), lambda: ("s", a, rng.uniform(0.05, 0.3)),
                lambda: ("d", b, _disc(rng, 1.0)), lambda: ("r", a, rng.uniform(-PI, PI)),
                lambda: ("s", b, rng.uniform(-0.3, -0.05)), lambda: ("bs", a, b, theta())]
        return [turn[i % len(turn)]() for i in range(case["gates"])]
    if case["mix"] == "transfer":
        o, ops = len(regs) - 1, []
        for q in range(case["gates"] // 3):
            ops += [("cd", o, q, 0, _disc(rng, 1.0)), ("h", q, 0), ("cr", o, q, 0, rng.uniform(-PI, PI))]
        return ops
    a, b = osc
    ops = [("h", 0, 0), ("d", a, _disc(rng, 1.0)), ("cd", b, 0, 0, _disc(rng, 1.0)), ("r", a, rng.uniform(-PI, PI)),
           ("cr", b, 0, 0, rng.uniform(-0.75, 0.75)), ("s", b, rng.uniform(-0.3, 0.3)),
           ("cs", a, 0, 0, rng.uniform(0.05, 0.3)), ("bs", a, b, rng.uniform(-1.4, 1.4)),
           ("cbs", a, b, 0, 0, rng.uniform(-1.4, 1.4)), ("q1q2", a, b, rng.uniform(-0.3, 0.3)),
           ("sheer", a, rng.uniform(-0.3, 0.3)), ("phaseCubic", b, rng.uniform(-0.05, 0.05)),
           ("rx", 0, 0, rng.uniform(-PI, PI)), ("ry", 0, 0, rng.uniform(-PI, PI)), ("rz", 0, 0, rng.uniform(-PI, PI)),
           ("x", 0, 0), ("p", a), ("cp", b, 0, 0), ("ftQ2P", a), ("sheer", a, rng.uniform(-0.2, 0.2)), ("ftP2Q", a)]
    ops.append(("swap", a, b) if regs[a] == regs[b] else ("z", 0, 0))
    return ops[:case["gates"]]


def _inits(case, seed):
    """Per register: ("zero",) for qubits, ("cat", [(alpha, coefficient), ...]) for oscillators."""
    rng, out = random.Random(1000003 * seed + 29), []
    for n in _regs(case):
        if n < 4:
            out.append(("zero",))
            continue
        k = 3 if case["mix"] == "transfer" else 1
        out.append(("cat", [(_disc(rng, 1.5), complex(rng.gauss(0, 1), rng.gauss(0, 1)) if k > 1 else 1.0)
                            for _ in range(k)]))
    return out


def _prepare_circuit(case, seed):
    regs = _regs(case)
    sep = SeparableState(regs)
    for r, i in enumerate(_inits(case, seed)):
        if i[0] == "zero":
            sep.setZero(r)
        else:
            sep.setCat(r, i[1])
    h = HipCvdv(regs, precision=case["prec"])
    ops, graph = _ops(case, seed), None
    if case["graph"]:
        h.initStateVector(sep)
        with h.capture() as graph:
            _apply(h, ops)
    return {"case": case, "h": h, "sep": sep, "ops": ops, "graph": graph}


def _apply(h, ops):
    for op in ops:
        getattr(h, op[0])(*op[1:])


def _measured(case):
    """What the program measures: the qubits (jointly in a state transfer)."""
    regs = _regs(case)
    return list(range(len(regs) - 1)) if case["mix"] == "transfer" else [0]


def _run_circuit(s):
    h, case = s["h"], s["case"]
    h.initStateVector(s["sep"])
    if s["graph"] is not None:
        s["graph"].launch()
    else:
        _apply(h, s["ops"])
    probs, state = h.m(*_measured(case)), h.getStateTensor()
    if case["prec"] == "mixed":
        return {"state": state.to(torch.complex64), "probs": probs.astype(np.float32)}
    return {"state": state, "probs": probs}


# register Fourier transforms that a gate's definition holds
_FTS = {"d": 2, "cd": 2, "r": 2, "cr": 2, "s": 4, "cs": 4, "bs": 4, "cbs": 4, "ftQ2P": 1, "ftP2Q": 1}


def _work_circuit(case):
    regs = _regs(case)
    size = 2.0 ** sum(regs)
    amp = 8 if case["prec"] == "mixed" else 16
    osc = max(regs)
    gates = [op[0] for op in _ops(case, 0)]
    # each gate reads and writes the state once; the result is written once and
    # read once for the measurement
    bytes_ = size * amp * 2 * len(gates) + size * amp * 2
    flops = size * sum(5.0 * osc * _FTS.get(g, 0) + 12.0 for g in gates)
    return {"bytes": bytes_, "flops": flops}


# ---------------------------------------------------------------- batches
def _sweep(case, seed):
    """Circuits (shape, alpha, gates): 1 to 3 qubits and an oscillator of 2^8 to 2^12
    points, 50 to 200 gates each.  Shapes and gate kinds are the case's, parameters the seed's."""
    fixed, rng, out = random.Random(4), random.Random(1000003 * seed + 31), []
    for _ in range(case["circuits"]):
        q, n = fixed.randint(1, 3), fixed.randint(8, 12)
        gates = []
        for _ in range(fixed.randint(50, 200)):
            k, b = fixed.randrange(7), fixed.randrange(q)
            gates.append([("h", 0, b), ("rx", 0, b, rng.uniform(-PI, PI)), ("rz", 0, b, rng.uniform(-PI, PI)),
                          ("cd", 1, 0, b, _disc(rng, 0.5)), ("r", 1, rng.uniform(-PI, PI)),
                          ("s", 1, rng.uniform(-0.3, 0.3)), ("cp", 1, 0, b)][k])
        out.append(([q, n], _disc(rng, 2.0), gates))
    return out


def _qubits_zero(q):
    a = np.zeros(1 << q, dtype=np.complex128)
    a[0] = 1.0
    return a


def _coherent(n, alpha):
    size = 1 << n
    dx = math.sqrt(2 * PI / size)
    x = (np.arange(size) - (size - 1) * 0.5) * dx
    q, p = math.sqrt(2) * alpha.real, math.sqrt(2) * alpha.imag
    return PI ** -0.25 * math.sqrt(dx) * np.exp(-0.5 * (x - q) ** 2) * np.exp(1j * (p * x - 0.5 * p * q))


def _prepare_batch(case, seed):
    circuits = _sweep(case, seed)
    b = HipCvdvBatch([c[0] for c in circuits], precision=case["prec"])
    for i, (_, _, gates) in enumerate(circuits):
        _apply(b.circuit(i), gates)
    b.initFromSeparable([[_qubits_zero(s[0]), _coherent(s[1], alpha)] for s, alpha, _ in circuits])
    b.autotune(1)
    return {"case": case, "batch": b}


def _run_batch(s):
    b = s["batch"]
    b.run()
    out = {"qubits": np.concatenate(b.measure(0)), "modes": np.concatenate(b.measure(1)), "norms": b.norms()}
    if s["case"]["prec"] == "mixed":
        return {k: v.astype(np.float32) for k, v in out.items()}
    return out


def _work_batch(case):
    amp = 8 if case["prec"] == "mixed" else 16
    bytes_ = flops = 0.0
    for (q, n), _, gates in _sweep(case, 0):
        size = 2.0 ** (q + n)
        bytes_ += 2 * size * amp + 16 * 2.0 ** n
        flops += size * sum(5.0 * n * _FTS.get(g[0], 0) + 12.0 for g in gates)
    return {"bytes": bytes_, "flops": flops}


# ---------------------------------------------------------------- loaded states
def _slices(case, seed):
    """An entangled state of unit norm: every value of the other registers carries its own
    superposition of two coherent states of the largest register.  (slices, points), complex128."""
    regs, rng = _regs(case), random.Random(1000003 * seed + 37)
    n = max(regs)
    others = 1 << (sum(regs) - n)
    k = min(others, 64)
    rows = []
    for _ in range(k):
        w = [complex(rng.gauss(0, 1), rng.gauss(0, 1)) for _ in range(2)]
        rows.append(w[0] * _coherent(n, _disc(rng, 2.0)) + w[1] * _coherent(n, _disc(rng, 2.0)))
    base = torch.from_numpy(np.array(rows))
    # more slices than that mix the first ones with a seeded unitary-like weight
    g = torch.Generator().manual_seed(1000003 * (seed % 1000000) + 41)
    if others > k:
        mix = torch.randn(others, k, 2, generator=g, dtype=torch.float64)
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        base = torch.view_as_complex(mix).to(dev) @ base.to(dev)
    return base / torch.linalg.vector_norm(base)


def _target(case):
    regs = _regs(case)
    return regs.index(max(regs))


def _flat(case, seed):
    """The same state in the flat order of the registers."""
    regs, t = _regs(case), _target(case)
    x = _slices(case, seed)
    lead = 1 << sum(regs[:t])
    return x.reshape(lead, -1, 1 << regs[t]).transpose(1, 2).contiguous().reshape(-1)


def _prepare_loaded(case, seed):
    h = HipCvdv(_regs(case), precision=case["prec"])
    h.initFromArray(_flat(case, seed).to("cuda"))
    s = {"case": case, "h": h, "reg": _target(case)}
    if case["kind"] == "grid":
        s["xs"], s["ps"] = _window(case, seed)
    if case["kind"] == "readouts":
        regs, rng = _regs(case), random.Random(1000003 * seed + 43)
        s["sep"] = SeparableState(regs)
        s["other"] = HipCvdv(regs, precision=case["prec"])
        s["other"].initFromArray(_flat(case, seed + 500009).to("cuda"))
        s["alphas"] = [_disc(rng, 1.0) for _ in regs]
        for r, n in enumerate(regs):
            if n < 4:
                s["sep"].setUniform(r)
            else:
                s["sep"].setCoherent(r, s["alphas"][r])
    return s


def _loaded(case, seed):
    """What the simulator holds after loading: rounded once to its amplitudes' width."""
    x = _flat(case, seed)
    return x.to(torch.complex64).to(torch.complex128) if case["prec"] == "mixed" else x


# native grids
def _run_native(s):
    h, out = s["h"], {}
    if s["case"]["wigner"]:
        out["wigner"] = h.getWigner(s["reg"], device=True)
    if s["case"]["husimi"]:
        out["husimi"] = h.getHusimiQ(s["reg"], device=True)
    return out


def _work_native(case):
    regs = _regs(case)
    n = max(regs)
    size, points, slices = 2.0 ** sum(regs), 4.0 ** n, 2.0 ** (sum(regs) - n)
    amp = 8 if case["prec"] == "mixed" else 16
    bytes_ = flops = 0.0
    if case["wigner"]:
        # a real transform of each row of pair products; half the pairs determine it
        bytes_ += size * amp + points * 8
        flops += points * (4.0 * slices + 2.5 * n)
    if case["husimi"]:
        bytes_ += size * amp + points * 8
        flops += points * slices * (5.0 * n + 5.0)
    return {"bytes": bytes_, "flops": flops}


# windows of phase space
def _window(case, seed):
    rng = random.Random(1000003 * seed + 47)
    c = [rng.uniform(-0.5, 0.5) for _ in range(2)]
    return (c[0] + np.linspace(-6.0, 6.0, case["points"]), c[1] + np.linspace(-6.0, 6.0, case["points"]))


def _run_grid(s):
    h, case = s["h"], s["case"]
    return {"wigner": h.getWignerGrid(s["reg"], s["xs"], s["ps"], per_slice=case["branches"], native=case["native"]),
            "husimi": h.getHusimiQGrid(s["reg"], s["xs"], s["ps"], per_slice=case["branches"])}


def _work_grid(case):
    regs = _regs(case)
    n = max(regs)
    size, slices, k = 2.0 ** sum(regs), 2.0 ** (sum(regs) - n), float(case["points"])
    amp = 8 if case["prec"] == "mixed" else 16
    pictures = slices if case["branches"] else 1.0
    bytes_ = 2 * size * amp + 2 * pictures * k * k * 8
    # Wigner: per point a real sum over the 2^n numbers of a Hermitian row, after an interpolation
    # of each slice at each x; Husimi: per slice and point a complex sum over the 2^n grid points
    flops = pictures * k * k * 2.0 * 2.0 ** n + slices * k * 5.0 * n * 2.0 ** n + slices * k * k * 8.0 * 2.0 ** n
    return {"bytes": bytes_, "flops": flops}


# readouts that leave the state as it is
def _run_readouts(s):
    h, case = s["h"], s["case"]
    out = {"norm": h.m(), "m0": h.m(0), "m1": h.m(1), "m2": h.m(2), "m12": h.m(1, 2), "m20": h.m(2, 0),
           "m012": h.m(0, 1, 2), "product": h.getFidelity(s["sep"]), "overlap": h.fidelityWith(s["other"]),
           "photons": h.getPhotonNumber(s["reg"])}
    if case["prec"] == "mixed":  # the transform of a photon number is in the amplitudes' width
        return {k: np.asarray(v, dtype=np.float32) for k, v in out.items()}
    return {k: np.asarray(v, dtype=np.float64) for k, v in out.items()}


def _work_readouts(case):
    regs = _regs(case)
    size = 2.0 ** sum(regs)
    amp = 8 if case["prec"] == "mixed" else 16
    bytes_ = size * amp * (10 + 1 + 4) + 8 * (2 * size)
    return {"bytes": bytes_, "flops": size * (9 * 4.0 + 20.0 + 2 * 5.0 * max(regs))}


# ---------------------------------------------------------------- the interface
def prepare(case, seed):
    if case["kind"] == "circuit":
        return _prepare_circuit(case, seed)
    if case["kind"] == "batch":
        return _prepare_batch(case, seed)
    return _prepare_loaded(case, seed)


def run(state):
    return {"circuit": _run_circuit, "batch": _run_batch, "native": _run_native, "grid": _run_grid,
            "readouts": _run_readouts}[state["case"]["kind"]](state)


def work(case):
    return {"circuit": _work_circuit, "batch": _work_batch, "native": _work_native, "grid": _work_grid,
            "readouts": _work_readouts}[case["kind"]](case)


# ---------------------------------------------------------------- the same in 64 bits
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _odd(n):
    """The odd integers m = 2 j - N + 1 of the grid points x_j = m dx / 2."""
    return 2 * torch.arange(1 << n, device=_dev(), dtype=torch.int64) - (1 << n) + 1


def _unit(angle):
    return torch.polar(torch.ones_like(angle), angle)


class _Plain:
    """Every gate on a complex128 tensor with one axis per register."""

    def __init__(self, regs, psi):
        self.regs, self.psi = regs, psi.reshape([1 << n for n in regs])
        self.dx = [math.sqrt(2 * PI / (1 << n)) for n in regs]

    def x(self, r):
        return _odd(self.regs[r]).to(torch.float64) * (0.5 * self.dx[r])

    def along(self, v, r):
        shape = [1] * len(self.regs)
        shape[r] = -1
        return v.reshape(shape)

    def sign(self, reg, qubit):
        """+1 where the control qubit is 0, -1 where it is 1."""
        n = self.regs[reg]
        j = torch.arange(1 << n, device=_dev())
        return self.along(1.0 - 2.0 * ((j >> (n - 1 - qubit)) & 1).to(torch.float64), reg)

    def phase(self, r, f, ctrl=None):
        a = self.along(f(self.x(r)), r)
        if ctrl is not None:
            a = a * self.sign(*ctrl)
        self.psi *= _unit(a)

    def product(self, r1, r2, c, ctrl=None):
        a = c * self.along(self.x(r1), r1) * self.along(self.x(r2), r2)
        if ctrl is not None:
            a = a * self.sign(*ctrl)
        self.psi *= _unit(a)

    def ft(self, r, inverse=False):
        # N^-1/2 exp(-+2 pi i m_j m_k / 4N) = (phase of m_k) DFT (phase of m_j) (constant), reduced in integers
        n = self.regs[r]
        size = 1 << n
        s = -1.0 if inverse else 1.0
        t = self.along(_unit(s * 2 * PI * torch.remainder((size - 1) * _odd(n), 4 * size).to(torch.float64)
                             / (4 * size)), r)
        c = cmath.exp(s * 2j * PI * (((size - 1) * (size - 1)) % (4 * size)) / (4 * size))
        self.psi *= t
        self.psi = (torch.fft.ifft if inverse else torch.fft.fft)(self.psi, dim=r, norm="ortho")
        self.psi *= t * c

    def matrix(self, reg, qubit, m):
        n = self.regs[reg]
        shape = list(self.psi.shape)
        v = self.psi.reshape(shape[:reg] + [1 << qubit, 2, 1 << (n - 1 - qubit)] + shape[reg + 1:])
        a, b = v.select(reg + 1, 0), v.select(reg + 1, 1)
        self.psi = torch.stack([m[0][0] * a + m[0][1] * b, m[1][0] * a + m[1][1] * b], reg + 1).reshape(shape)

    def rot(self, reg, qubit, axis, t):
        c, s = math.cos(t / 2), math.sin(t / 2)
        self.matrix(reg, qubit, {"x": [[c, -1j * s], [-1j * s, c]], "y": [[c, -s], [s, c]],
                                 "z": [[cmath.exp(-0.5j * t), 0], [0, cmath.exp(0.5j * t)]]}[axis])

    def h(self, r, q):
        w = math.sqrt(0.5)
        self.matrix(r, q, [[w, w], [w, -w]])

    def x_(self, r, q):
        self.rot(r, q, "x", PI)

    def z(self, r, q):
        self.rot(r, q, "z", PI)

    def rx(self, r, q, t):
        self.rot(r, q, "x", t)

    def ry(self, r, q, t):
        self.rot(r, q, "y", t)

    def rz(self, r, q, t):
        self.rot(r, q, "z", t)

    def p(self, r):
        self.psi = torch.flip(self.psi, [r])

    def cp(self, t, c, q):
        one = (self.sign(c, q) < 0).expand(self.psi.shape)
        self.psi = torch.where(one, torch.flip(self.psi, [t]), self.psi)

    def swap(self, a, b):
        self.psi = self.psi.transpose(a, b).contiguous()

    def sheer(self, r, t):
        self.phase(r, lambda x: t * x * x)

    def phaseCubic(self, r, t):
        self.phase(r, lambda x: t * x * x * x)

    def q1q2(self, a, b, c):
        self.product(a, b, c)

    def ftQ2P(self, r):
        self.ft(r)

    def ftP2Q(self, r):
        self.ft(r, True)

    def d(self, r, a, ctrl=None):
        if abs(a.imag) > 1e-12:
            self.phase(r, lambda x: math.sqrt(2) * a.imag * x, ctrl)
        if abs(a.real) > 1e-12:
            self.ft(r)
            self.phase(r, lambda x: -math.sqrt(2) * a.real * x, ctrl)
            self.ft(r, True)

    def cd(self, t, c, q, a):
        self.d(t, a, (c, q))

    def shears(self, r, t, ctrl=None):
        if abs(t) < 1e-15:
            return
        self.phase(r, lambda x: -0.5 * math.tan(t / 2) * x * x, ctrl)
        self.ft(r)
        self.phase(r, lambda x: -0.5 * math.sin(t) * x * x, ctrl)
        self.ft(r, True)
        self.phase(r, lambda x: -0.5 * math.tan(t / 2) * x * x, ctrl)

    def r(self, r, t):
        k = int(np.rint(t / (PI / 2)))
        if k % 4 == 1:
            self.ft(r)
        elif k % 4 == 2:
            self.p(r)
        elif k % 4 == 3:
            self.ft(r, True)
        self.shears(r, t - k * (PI / 2))

    def cr(self, t, c, q, a):
        k = int(np.rint(a / (PI / 2)))
        if k % 4 == 2:
            self.p(t)
            self.rz(c, q, PI)
        elif k % 4:
            self.ft(t, k % 4 == 3)
            self.cp(t, c, q)
            self.rz(c, q, PI / 2 if k % 4 == 1 else -PI / 2)
        self.shears(t, a - k * (PI / 2), (c, q))

    def s(self, r, v):
        up, dn, w = math.exp(0.5 * v), math.exp(-0.5 * v), math.sqrt(abs(math.exp(v) - 1.0))
        g = 1.0 if v >= 0 else -1.0
        for c, inv in ((-0.5 * up * w, False), (0.5 * dn * w * g, True), (0.5 * dn * w, False),
                       (-0.5 * up * w * g, True)):
            # momentum shears under a transform, position shears between them
            self.ft(r, inv)
            self.phase(r, lambda x, c=c: c * x * x)

    def cs(self, t, c, q, v):
        ch, sh, w = math.cosh(v), math.sinh(v), math.sqrt(2 * abs(math.sinh(0.5 * v)))
        ctl = (c, q)
        self.sheer(t, 0.5 * w * ch)
        self.phase(t, lambda x: -0.5 * w * sh * x * x, ctl)
        self.ft(t)
        self.sheer(t, 0.5 * (ch - 1) / w)
        self.phase(t, lambda x: 0.5 * sh / w * x * x, ctl)
        self.ft(t, True)
        self.sheer(t, -0.5 * w)
        self.ft(t)
        self.sheer(t, 0.5 * (ch - 1) / w)
        self.phase(t, lambda x: -0.5 * sh / w * x * x, ctl)
        self.ft(t, True)

    def bs(self, a, b, t, ctrl=None):
        k = int(math.copysign(math.floor(abs(t / PI) + 0.5), t))
        if k % 4 == 2:
            self.p(a)
            self.p(b)
        elif k % 4:
            self.ft(a, k % 4 == 3)
            self.ft(b, k % 4 == 3)
            self.swap(a, b)
        t -= k * PI
        if abs(t) < 1e-15:
            return
        cq, cp = -math.tan(0.25 * t), -math.sin(0.5 * t)
        self.product(a, b, cq, ctrl)
        self.ft(a)
        self.ft(b)
        self.product(a, b, cp, ctrl)
        self.ft(a, True)
        self.ft(b, True)
        self.product(a, b, cq, ctrl)

    def cbs(self, a, b, c, q, t):
        self.bs(a, b, t, (c, q))  # |t| < pi / 2 here: no half turns

    def apply(self, ops):
        for op in ops:
            getattr(self, {"x": "x_"}.get(op[0], op[0]))(*op[1:])

    def marginal(self, *keep):
        p = self.psi.real.square() + self.psi.imag.square()
        drop = [i for i in range(len(self.regs)) if i not in keep]
        p = p.sum(dim=drop) if drop else p
        order = sorted(keep)
        return p.permute([order.index(k) for k in keep]) if keep else p


def _start(case, seed):
    psi = torch.ones(1, dtype=torch.complex128, device=_dev())
    for n, i in zip(_regs(case), _inits(case, seed)):
        if i[0] == "zero":
            a = _qubits_zero(n)
        else:
            a = sum(c * _coherent(n, al) for al, c in i[1])
            a = a / np.linalg.norm(a)
        psi = torch.outer(psi, torch.from_numpy(np.asarray(a, dtype=np.complex128)).to(_dev())).reshape(-1)
    return psi


def _exact_circuit(case, seed):
    p = _Plain(_regs(case), _start(case, seed))
    p.apply(_ops(case, seed))
    return {"state": p.psi.reshape(-1), "probs": p.marginal(*_measured(case))}


def _exact_batch(case, seed):
    qubits, modes, norms = [], [], []
    for shape, alpha, gates in _sweep(case, seed):
        a = np.outer(_qubits_zero(shape[0]), _coherent(shape[1], alpha)).reshape(-1)
        p = _Plain(shape, torch.from_numpy(a).to(_dev()))
        p.apply(gates)
        qubits.append(p.marginal(0))
        modes.append(p.marginal(1))
        norms.append(qubits[-1].sum())
    return {"qubits": torch.cat(qubits), "modes": torch.cat(modes), "norms": torch.stack(norms)}


def _rows(case, seed):
    """The loaded state as (slices, points) of the target register."""
    regs, t = _regs(case), _target(case)
    n, lead = regs[t], 1 << sum(regs[:t])
    v = _loaded(case, seed).to(_dev()).reshape(lead, 1 << n, -1)
    return v.transpose(1, 2).reshape(-1, 1 << n).contiguous()


def _exact_native(case, seed):
    x, out = _rows(case, seed), {}
    size = x.shape[1]
    dx = math.sqrt(2 * PI / size)
    j = torch.arange(size, device=_dev())
    if case["wigner"]:
        half = (size - 1) // 2
        rho = x.transpose(0, 1).contiguous() @ x.conj().resolve_conj()
        k = j[None, :] - half
        lo, hi = j[:, None] - k, j[:, None] + k
        inside = (lo >= 0) & (lo < size) & (hi >= 0) & (hi < size)
        g = torch.where(inside, rho[lo.clamp(0, size - 1), hi.clamp(0, size - 1)], torch.zeros_like(rho[0, 0]))
        g = torch.fft.ifft(g, dim=1, norm="forward")
        g = torch.roll(g, size // 2, dims=1).transpose(0, 1)
        turn = -PI * torch.remainder((size - 1) * (j - size // 2), 2 * size).to(torch.float64) / size
        out["wigner"] = ((g * _unit(turn)[:, None]).real * (dx / PI)).contiguous()
        del rho, g
    if case["husimi"]:
        d = (j[None, :] - j[:, None]).to(torch.float64) * dx
        w = PI ** -0.25 * math.sqrt(dx) * torch.exp(-0.5 * d * d)
        q = torch.zeros((size, size), dtype=torch.float64, device=_dev())
        for row in x:
            f = torch.fft.fft(w * row[None, :], dim=1)
            q += f.real.square() + f.imag.square()
        out["husimi"] = (torch.roll(q, size // 2, dims=1).transpose(0, 1) / PI).contiguous()
    return out


def _exact_grid(case, seed):
    v = _rows(case, seed)
    slices, size = v.shape
    dx = math.sqrt(2 * PI / size)
    xs, ps = (torch.from_numpy(a).to(_dev()) for a in _window(case, seed))
    # Wigner: x = x_i + t dx, each slice interpolated by its own trigonometric polynomial
    u = xs / dx + 0.5 * (size - 1)
    near = torch.round(u)
    i = torch.where((u - near).abs() < 1e-9, near, torch.floor(u))
    t = torch.where((u - near).abs() < 1e-9, torch.zeros_like(u), u - i)
    i = i.to(torch.int64)
    k = torch.fft.fftfreq(size, 1.0 / size, device=_dev(), dtype=torch.float64)
    spec = torch.fft.fft(v, dim=1)
    half = size // 2
    d = torch.arange(-half, half + 1, device=_dev())
    lo, hi = i[:, None] - d, i[:, None] + d
    inside = (lo >= 0) & (lo < size) & (hi >= 0) & (hi < size)
    m = (2 * d - 1 if case["native"] else 2 * d).to(torch.float64)
    e = _unit(dx * ps[:, None] * m[None, :])
    wig, rows = [], torch.arange(len(xs), device=_dev())[:, None]
    for s in range(slices):
        phi = torch.fft.ifft(spec[s][None, :] * _unit(2 * PI * t[:, None] * k[None, :] / size), dim=1)
        a = phi[rows, lo.clamp(0, size - 1)] * phi[rows, hi.clamp(0, size - 1)].conj()
        a = torch.where(inside, a, torch.zeros_like(a))
        wig.append((e @ a.transpose(0, 1).contiguous()).real * (dx / PI))
    # Husimi: per slice the overlap with a displaced Gaussian
    x = _odd(int(size).bit_length() - 1).to(torch.float64) * (0.5 * dx)
    win = torch.exp(-0.5 * (x[None, :] - xs[:, None]) ** 2)
    e = _unit(-ps[:, None] * x[None, :])
    hus = []
    for s in range(slices):
        f = e @ (win * v[s][None, :]).transpose(0, 1).contiguous()
        hus.append((f.real.square() + f.imag.square()) * (dx / PI ** 1.5))
    wig, hus = torch.stack(wig), torch.stack(hus)
    return {"wigner": wig if case["branches"] else wig.sum(0), "husimi": hus if case["branches"] else hus.sum(0)}


def _exact_readouts(case, seed):
    regs = _regs(case)
    p = _Plain(regs, _loaded(case, seed).to(_dev()))
    other = _loaded(case, seed + 500009).to(_dev())
    rng = random.Random(1000003 * seed + 43)
    sep = torch.ones(1, dtype=torch.complex128, device=_dev())
    for n in regs:
        alpha = _disc(rng, 1.0)
        a = np.full(1 << n, 2.0 ** (-n / 2), dtype=np.complex128) if n < 4 else _coherent(n, alpha)
        sep = torch.outer(sep, torch.from_numpy(np.asarray(a, dtype=np.complex128)).to(_dev())).reshape(-1)
    out = {"norm": p.marginal(0).sum(), "m0": p.marginal(0), "m1": p.marginal(1), "m2": p.marginal(2),
           "m12": p.marginal(1, 2), "m20": p.marginal(2, 0), "m012": p.marginal(0, 1, 2),
           "product": torch.vdot(p.psi.reshape(-1), sep).abs().square(),
           "overlap": torch.vdot(p.psi.reshape(-1), other.reshape(-1)).abs().square()}
    t = _target(case)
    x2 = p.x(t).square()
    q2 = (p.marginal(t) * x2).sum()
    p.ft(t)
    out["photons"] = (q2 + (p.marginal(t) * x2).sum() - 1.0) / 2.0
    return out


def exact(case, seed):
    return {"circuit": _exact_circuit, "batch": _exact_batch, "native": _exact_native, "grid": _exact_grid,
            "readouts": _exact_readouts}[case["kind"]](case, seed)
