"""Spectra above 4 GB: the fused x pass with 64-bit offsets (512, 768 and 1024
points), the mixed-radix fused pass (other lengths) and, on the other side of the
comparison, the stage sequence, whose x columns run mixed-radix there.  Fields are
drawn on the device.

FP64: 1e-9 per bin, as the other comparisons of the two forms, and Parseval: the
zero lag is the mean square, to 1e-12 log2(cells).  FP32 and mixed storage
against FP64 on the same grid by the 2-norm over all bins: 32 roundings of 2^-24
(FP32: log2 N stages, product and inverse) and 16 (mixed: three passes of stores
and exchanges, doubled by the product)."""
import ctypes

import numpy as np
import pytest

from fftcorr_amd import _lib
from fftcorr_amd.correlate import Correlator, PeriodicCorrelator
from gpu_helpers import floor_rel_err

pytestmark = pytest.mark.gpu

CELL = 2.0


def field(shape, precision, seed):
    """Relative overdensity of 20 million random points, nearest cell."""
    g = _lib.DeviceGrid(shape, cell_size=CELL, precision=precision)
    st = _lib.MaStats()
    _lib.check(_lib.lib().fc_add_random_particles(g.handle, 20_000_000, 1.0, 0, 1, None, seed,
                                                  20_000_000, ctypes.byref(st)))
    g.normalize(st.totw / float(np.prod(shape)))
    return g


def correlate(shape, precision, algorithm, mode, a, b=None):
    # 13^3 lags, 31 wavenumbers along the longest axis.
    kmax = 15.5 * 2 * np.pi / (CELL * max(shape))
    args = (0, 6 * CELL, CELL, kmax, kmax / 8, 4)
    if mode == "yamamoto":
        c = Correlator(shape, CELL, [900.0, -700.0, 40.0], *args, precision=precision)
    else:
        c = PeriodicCorrelator(shape, CELL, *args, precision=precision)
    c.algorithm = algorithm
    lib = _lib.lib()
    if mode == "interlaced":
        _lib.check(lib.fc_corr_autocorrelate_interlaced(c._handle, a.handle, b.handle))
    elif mode == "cross":
        _lib.check(lib.fc_corr_set_grid2(c._handle, b.handle))
        _lib.check(lib.fc_corr_cross_correlate(c._handle, a.handle))
    else:
        _lib.check(lib.fc_corr_autocorrelate(c._handle, a.handle))
    c._fetch()
    return c.results()


@pytest.mark.parametrize("shape,mode", [
    ((1024, 1024, 512), "auto"), ((1024, 1024, 512), "yamamoto"),
    ((1024, 1024, 512), "cross"), ((1024, 1024, 512), "interlaced"),
    ((768, 1408, 512), "interlaced"), ((512, 2048, 512), "cross"), ((2048, 512, 512), "auto"),
    ((2048, 512, 512), "interlaced"), ((1250, 864, 500), "cross")])
def test_fused_matches_plain_fp64(shape, mode):
    a = field(shape, "fp64", 11)
    b = field(shape, "fp64", 12) if mode in ("cross", "interlaced") else None
    got = correlate(shape, "fp64", "fused", mode, a, b)
    want = correlate(shape, "fp64", "plain", mode, a, b)
    for key in ("r_counts", "k_counts"):
        np.testing.assert_array_equal(got[key], want[key])
    for key in ("r_hist", "k_hist"):
        assert floor_rel_err(got[key], want[key]).max() < 1e-9, key
    if mode == "auto":
        ncells = float(np.prod(shape))
        mean_sq = a.stats()[1] / ncells
        assert abs(got["zerolag"] - mean_sq) < 1e-12 * np.log2(ncells) * mean_sq


@pytest.mark.parametrize("precision,roundings", [("fp32", 32), ("mixed", 16)])
def test_fp32_storage_matches_fp64(precision, roundings):
    shape = (1024, 1024, 1024)
    a = field(shape, "fp32", 13)
    want = correlate(shape, "fp64", "plain", "auto", a)
    got = correlate(shape, precision, "fused", "auto", a)
    for key in ("r_counts", "k_counts"):
        np.testing.assert_array_equal(got[key], want[key])
    for key in ("r_hist", "k_hist"):
        off = np.linalg.norm(got[key] - want[key])
        assert off < roundings * 2.0 ** -24 * np.linalg.norm(want[key]), key
