"""Mixed-radix transforms (csrc/fft_gen*): lengths without a compile-time
plan against numpy, at every radix, at single-stage and many-stage lengths, at
chirp-convolution lengths and with odd row counts (rows are transformed in
pairs); the fused x pass of such lengths against the stage-by-stage form.
Tolerances as tests/test_gpu_fft.py: FP64 1e-12 log2(N), FP32 3e-6 log2(N) of
the largest value."""
import numpy as np
import pytest

from fftcorr_amd.correlate import Correlator, PeriodicBatch, PeriodicCorrelator
from fftcorr_amd.grid import ConfigSpaceGrid
from gpu_helpers import fft_c2r, fft_r2c, floor_rel_err

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-12, "fp32": 3e-6}
# Each axis in turn takes: a single butterfly of every radix (1 .. 15), two
# and three stages, lengths whose only plan has idle threads, and
# lengths with a factor above 13 (17, 101, 2 * 31, 509).
SHAPES = [(2, 3, 1), (5, 7, 9), (10, 11, 13), (15, 12, 6), (6, 10, 15), (7, 9, 11), (13, 5, 3),
          (26, 33, 35), (121, 45, 20), (100, 36, 250), (3, 169, 243), (17, 62, 101), (101, 17, 31),
          (2, 400, 400), (400, 3, 22), (3, 2, 1000), (4, 1250, 5), (1250, 2, 34), (2, 509, 3),
          (3, 3, 509), (1, 3, 2)]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", SHAPES)
def test_transforms_match_numpy(shape, precision):
    rng = np.random.default_rng(sum(shape))
    a = rng.normal(size=shape)
    tol = TOL[precision] * np.log2(max(a.size, 2))
    ref = np.fft.rfftn(a)
    err = np.max(np.abs(fft_r2c(a, precision) - ref)) / np.max(np.abs(ref))
    assert err <= tol, err
    back = np.fft.irfftn(ref, s=shape, axes=(0, 1, 2), norm="forward")
    err = np.max(np.abs(fft_c2r(ref, shape, precision) - back)) / np.max(np.abs(back))
    assert err <= tol, err


ARGS = (5.0, 2, 40.0, 5.0, 0.3, 0.02, 4)


@pytest.mark.parametrize("shape", [(20, 18, 21), (45, 20, 10), (36, 17, 30), (13, 24, 26)])
@pytest.mark.parametrize("mode", ["auto", "cross", "interlaced", "yamamoto"])
def test_fused_x_matches_plain(shape, mode):
    """FP64: the fused x pass against the stage sequence (the same operations
    in another order: 1e-9 per bin as the other parity bars).  Mixed against
    FP64 by the 2-norm over all bins: a value is rounded to FP32 at most eight
    times on its way to the power (grid, two exchanges and a store in each of
    the z and y passes, one load), the product doubles that: 16 x 2^-24 < 1e-6."""
    rng = np.random.default_rng(sum(shape))
    a, b = rng.normal(size=shape), rng.normal(size=shape)

    def run(precision, algorithm):
        if mode == "yamamoto":
            c = Correlator(shape, ARGS[0], [200.0, -50.0, 30.0], *ARGS[1:], precision=precision)
        else:
            c = PeriodicCorrelator(shape, *ARGS, precision=precision)
        c.algorithm = algorithm
        if mode == "interlaced":
            g = ConfigSpaceGrid.from_cell(shape, [0.0] * 3, ARGS[0], precision=precision)
            np.copyto(g.data, b)
            c.autocorrelate_interlaced(a, g)
        elif mode == "cross":
            c.cross_correlate(a, b)
        else:
            c.autocorrelate(a)
        return c.results()

    want = run("fp64", "plain")
    for precision in ("fp64", "mixed"):
        got = run(precision, "fused")
        for key in ("r_hist", "k_hist"):
            if precision == "fp64":
                assert floor_rel_err(got[key], want[key]).max() < 1e-9, key
            else:
                off = np.linalg.norm(got[key] - want[key])
                assert off < 1e-6 * np.linalg.norm(want[key]), key
        for key in ("r_counts", "k_counts"):
            np.testing.assert_array_equal(got[key], want[key])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_batch_members_equal_single(precision):
    """Odd member rows: a pair of rows never spans two members."""
    shape = (15, 9, 21)
    rng = np.random.default_rng(3)
    fields = [rng.normal(size=shape) for _ in range(3)]
    batch = PeriodicBatch(shape, *ARGS, nbatch=3, precision=precision)
    for i, f in enumerate(fields):
        batch.grid(i).upload(f)
    batch.autocorrelate()
    for i, f in enumerate(fields):
        c = PeriodicCorrelator(shape, *ARGS, precision=precision)
        c.autocorrelate(f)
        want, got = c.results(), batch.results(i)
        for key in ("r_hist", "k_hist", "r_counts", "k_counts"):
            np.testing.assert_array_equal(got[key], want[key], err_msg=key)
