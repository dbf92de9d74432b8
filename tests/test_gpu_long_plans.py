"""Compile-time plans of 3 2^a and of 1024 .. 4096 points: transforms against
numpy (columns with a ragged last tile, rows, every tile width the lengths
take) and the fused x pass against the stage-by-stage form.  Tolerances as
tests/test_gpu_fft.py (FP64 1e-12 log2(N), FP32 3e-6 log2(N) of the largest
value) and 1e-9 per bin in FP64."""
import numpy as np
import pytest

from fftcorr_amd.correlate import PeriodicCorrelator
from fftcorr_amd.grid import ConfigSpaceGrid
from gpu_helpers import fft_c2r, fft_r2c, floor_rel_err

pytestmark = pytest.mark.gpu

LENGTHS = [192, 384, 768, 1024, 1536, 2048, 3072, 4096]
TOL = {"fp64": 1e-12, "fp32": 3e-6}


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_transforms_match_numpy(n, axis, precision):
    shape = [2, 3, 36]
    shape[axis] = n
    rng = np.random.default_rng(n + axis)
    a = rng.normal(size=shape)
    tol = TOL[precision] * np.log2(a.size)
    ref = np.fft.rfftn(a)
    assert np.max(np.abs(fft_r2c(a, precision) - ref)) <= tol * np.max(np.abs(ref))
    back = np.fft.irfftn(ref, s=shape, axes=(0, 1, 2), norm="forward")
    assert np.max(np.abs(fft_c2r(ref, tuple(shape), precision) - back)) <= tol * np.max(np.abs(back))


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("mode", ["auto", "cross", "interlaced"])
@pytest.mark.parametrize("n", LENGTHS)
def test_fused_x_matches_plain(n, mode, precision):
    """FP32: the same transforms with other roundings; the 2-norm over all
    bins, 32 roundings of 2^-24 (log2 N stages, product and inverse)."""
    shape = (n, 6, 10)
    rng = np.random.default_rng(n)
    a, b = rng.normal(size=shape), rng.normal(size=shape)

    def run(algorithm):
        c = PeriodicCorrelator(shape, 5.0, 2, 40.0, 5.0, 0.3, 0.02, 4, precision=precision)
        c.algorithm = algorithm
        if mode == "interlaced":
            g = ConfigSpaceGrid.from_cell(shape, [0.0] * 3, 5.0, precision=precision)
            np.copyto(g.data, b)
            c.autocorrelate_interlaced(a, g)
        elif mode == "cross":
            c.cross_correlate(a, b)
        else:
            c.autocorrelate(a)
        return c.results()

    got, want = run("fused"), run("plain")
    for key in ("r_hist", "k_hist"):
        if precision == "fp64":
            assert floor_rel_err(got[key], want[key]).max() < 1e-9, key
        else:
            off = np.linalg.norm(got[key] - want[key])
            assert off < 32 * 2.0 ** -24 * np.linalg.norm(want[key]), key
    for key in ("r_counts", "k_counts"):
        np.testing.assert_array_equal(got[key], want[key])
