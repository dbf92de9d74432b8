"""Correlators of one context share the streams beside its own: interleaved calls,
calls from several threads and a correlator that ends between two calls of another
give the bits of a correlator alone."""
import ctypes
import threading

import numpy as np
import pytest

from fftcorr_amd import _lib
from fftcorr_amd.correlate import Correlator, PeriodicCorrelator

pytestmark = pytest.mark.gpu

KEYS = ("r_hist", "k_hist", "r_counts", "k_counts")


def make(kind, n, ctx):
    shape = (n, n, n)
    if kind == "survey":
        c = Correlator(shape, 5.0, [200.0, -50.0, 30.0], 2, 30.0, 5.0, 0.25, 0.02, 4)
    else:
        c = PeriodicCorrelator(shape, 5.0, 2, 30.0, 5.0, 0.25, 0.02, 4, context=ctx)
    return c, np.random.default_rng(n).normal(size=shape)


# 144^3: the k histogram runs beside the inverse; survey: three streams.
CASES = [("periodic", 144), ("survey", 40), ("periodic", 150), ("survey", 64)]


def alone(kind, n):
    c, a = make(kind, n, _lib.context())
    c.autocorrelate(a)
    return c.results()


def check(got, want):
    for key in KEYS:
        np.testing.assert_array_equal(got[key], want[key])


def test_interleaved_and_ended_between():
    want = [alone(*c) for c in CASES]
    live = [make(*c, _lib.context()) for c in CASES]
    for turn in range(3):
        for (c, a), w in zip(live, want):
            c.autocorrelate(a)
            check(c.results(), w)
        gone, a = make("survey", 48 + turn, _lib.context())
        gone.autocorrelate(a)
        del gone


def test_threads():
    want = [alone(*c) for c in CASES]
    live = [make(*c, _lib.context()) for c in CASES]
    bad = []

    def work(i):
        try:
            c, a = live[i]
            for _ in range(8):
                c.autocorrelate(a)
                check(c.results(), want[i])
        except BaseException as e:  # noqa: BLE001 -- reported below
            bad.append((CASES[i], e))

    th = [threading.Thread(target=work, args=(i,)) for i in range(len(CASES))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad


def test_work_spectra_are_allocated_once():
    """A survey correlator's work buffer has its full size (nine spectra for
    l <= 4) from set_grid2 on: the first correlation adds only the rest."""
    n = 64
    c, a = make("survey", n, _lib.context())
    spectrum = n * n * 40 * 16  # complex rows of 33 values padded to 40

    def held():
        now, full = ctypes.c_size_t(), ctypes.c_size_t()
        _lib.check(_lib.lib().fc_corr_footprint(c._handle, 0, ctypes.byref(now),
                                                ctypes.byref(full)))
        return now.value

    before = held()
    c.set_grid2(a)
    assert held() - before == (9 + 1) * spectrum  # and grid 2's own
    middle = held()
    c.cross_correlate(a)
    assert held() - middle < 8 * spectrum
