"""Large results copied to pageable host memory: every byte, at the edges of the chunks, for
two threads at a time, and again after the last context has been destroyed."""

import threading

import numpy as np
import pytest

from hipcvdv import HipCvdv

pytestmark = pytest.mark.gpu


def _loaded(regs, seed):
    rng = np.random.default_rng(seed)
    n = 1 << sum(regs)
    v = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    h = HipCvdv(regs)
    h.initFromArray(v)
    return h, v


# parts of 2^18 .. 2^21 numbers: below the chunked path, its smallest, and many chunks; the
# copied numbers are the loaded ones, so equality is exact
@pytest.mark.parametrize("regs", [[18], [1, 18], [1, 9, 10], [21]])
def test_state_bytes(regs):
    h, v = _loaded(regs, sum(regs))
    assert np.array_equal(h.getState(), v)


# a last chunk of a few bytes, whole chunks, a ragged last chunk; strips of columns stay below
# the chunked path, and a point's sum may be taken in another order there: 2^8 terms of
# magnitude <= 1 in FP64, 1e-12 of the largest value
@pytest.mark.parametrize("points", [725, 1024, 1100])
def test_grid_against_strips(points):
    h, _ = _loaded([1, 8], points)
    xs, ps = np.linspace(-6, 6, points), np.linspace(-5, 5, points)
    whole = h.getHusimiQGrid(1, xs, ps)
    strips = np.concatenate([h.getHusimiQGrid(1, x, ps) for x in np.array_split(xs, 5)], axis=1)
    assert whole.shape == strips.shape
    assert np.abs(whole - strips).max() <= 1e-12 * np.abs(strips).max()


def test_two_threads_and_a_later_context():
    pairs = [_loaded([20], 5), _loaded([1, 19], 6)]
    same = []

    def read(h, v):
        for _ in range(4):
            same.append(np.array_equal(h.getState(), v))

    threads = [threading.Thread(target=read, args=p) for p in pairs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert same == [True] * 8
    del pairs, threads
    h, v = _loaded([20], 7)
    assert np.array_equal(h.getState(), v)
