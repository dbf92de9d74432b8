"""Mass assignment at the edges of its tiles (8 x 32 target cells of an x
plane, 64 lanes that share a tile's particles) against the oracle."""
import numpy as np
import pytest

from fftcorr_amd.grid import ConfigSpaceGrid
from fftcorr_amd.particle_mesh import MassAssignor
from oracle import fftcorr_oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (2, 1, 3), (3, 7, 31), (4, 8, 32), (5, 9, 33), (3, 17, 64), (1, 2, 65)]


@pytest.mark.parametrize("scheme", [0, 1, 3])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("n", [1, 63, 65, 700])
def test_tile_edges(shape, scheme, n):
    rng = np.random.default_rng(n + 10 * sum(shape) + scheme)
    cell = 2.0
    ext = cell * np.array(shape)
    pos = rng.uniform(0, ext, size=(n, 3))
    # Half of them in one cell at the upper corner of the box, whose stencil
    # wraps on every axis: one key cell shared by many lanes.
    pos[n // 2:] = ext - rng.uniform(0.01, 0.9, size=(n - n // 2, 3))
    w = rng.uniform(0.5, 1.5, n)
    grids = []
    for _ in range(2):
        g = ConfigSpaceGrid(shape, [0, 0, 0], ext, cell_size=cell)
        MassAssignor(g, scheme, periodic_wrap=True).add_particles(pos, w)
        grids.append(g.data.copy())
    assert np.array_equal(grids[0], grids[1])
    x, ok = O.grid_coords(pos, np.zeros(3), cell, shape, True)
    ref = O.assign_mass(np.zeros(shape), x[ok], w[ok], scheme)
    # At most 27 n terms of one sign per cell, each with 6 roundings: 27 n + 6
    # units of 2^-53 for either side; cells that TSC reaches with a weight
    # near 0 by as many units of the largest 1D weight, 1.
    tol = 2 * (27 * n + 6) * 2.0 ** -53
    np.testing.assert_allclose(grids[0], ref, rtol=tol, atol=tol)
