"""Yamamoto transforms that share their launches (all m of one l, in one group,
in uneven groups, and on grids whose x pass runs in separate steps) against the
stage-by-stage sequence, one transform at a time."""
import numpy as np
import pytest

from fftcorr_amd.correlate import Correlator
from fftcorr_amd.grid import ConfigSpaceGrid

pytestmark = pytest.mark.gpu

# 256^3 and 250 x 300 x 200 hold 5 + 4 and 9 transforms of l = 4 in the group
# memory, 34 x 19 x 22 and 53 x 24 x 37 have a prime factor above 13 on one axis.
CASES = [((256, 256, 256), 4), ((250, 300, 200), 4), ((64, 32, 48), 1), ((64, 64, 64), 2),
         ((40, 36, 50), 3), ((34, 19, 22), 4), ((53, 24, 37), 4), ((8, 8, 8), 4)]


@pytest.mark.parametrize("shape,maxell", CASES)
def test_groups_match_single_transforms(shape, maxell):
    rng = np.random.default_rng(sum(shape) + maxell)
    cell = 5.0
    posmin = np.array([200.0, -100.0, -30.0])
    g = ConfigSpaceGrid.from_cell(shape, posmin, cell)
    g.data[:] = rng.normal(0.0, 1.0, shape)
    half = 0.4 * cell * min(shape)
    res = []
    for algo in ("plain", "fused"):
        c = Correlator(shape, cell, posmin, 2, half, half / 4, 0.3, 0.05, maxell)
        c.algorithm = algo
        c.autocorrelate(g)
        res.append(c.results())
    want, got = res
    for key in ("r_counts", "k_counts"):
        assert np.array_equal(want[key], got[key])
    # About 10 log2(N) 2^-53 of a transform's scale, the multipoles up to a
    # few hundred times smaller than the terms they cancel from.
    for key in ("r_hist", "k_hist"):
        scale = np.abs(want[key][0]).max()
        assert np.abs(want[key] - got[key]).max() <= 1e-11 * scale
    assert abs(want["zerolag"] - got["zerolag"]) <= 1e-12 * abs(want["zerolag"])
    # Again on the same correlator, and against the stored grid 2.
    again = c.autocorrelate(g) and c.results()
    assert np.array_equal(got["r_hist"], again["r_hist"])
    assert np.array_equal(got["k_hist"], again["k_hist"])
    c.cross_correlate(g)
    cross = c.results()
    assert np.abs(want["r_hist"] - cross["r_hist"]).max() <= 1e-11 * np.abs(want["r_hist"][0]).max()
