"""Host catalogues that reach the device in chunks, and the host copy of a
grid that was cleared on the device."""
import numpy as np
import pytest

from fftcorr_amd.grid import ConfigSpaceGrid
from fftcorr_amd.particle_mesh import MassAssignor

pytestmark = pytest.mark.gpu

MIB = 1 << 20
# Rows of 24 bytes around the length from which chunks are used (4 MiB), around
# whole chunks (2 MiB) and past every slot's first use (16 MiB), remainders of
# one row and of nearly a chunk among them.
ROWS = [4 * MIB // 24 - 1, 4 * MIB // 24 + 1, 6 * MIB // 24, 6 * MIB // 24 + 2,
        16 * MIB // 24 + 3, 40 * MIB // 24 - 5]


@pytest.mark.parametrize("n", ROWS)
def test_chunked_catalogue_arrives_whole(n):
    rng = np.random.default_rng(n)
    shape = (6, 5, 7)
    pos = rng.integers(0, shape, size=(n, 3)) + 0.5  # cell centres: counts are exact
    w = rng.integers(1, 9, n).astype(np.float64)
    g = ConfigSpaceGrid(shape, [0, 0, 0], shape, cell_size=1.0)
    ma = MassAssignor(g, 0)
    for _ in range(2):
        ma.add_particles(pos, w)
    cell = np.ravel_multi_index(tuple(pos.astype(int).T), shape)
    want = 2 * np.bincount(cell, weights=w, minlength=int(np.prod(shape))).reshape(shape)
    np.testing.assert_array_equal(g.data, want)
    assert ma.num_added == 2 * n and ma.totw == 2 * w.sum()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_clear_and_the_host_copy(precision):
    shape = (4, 4, 4)
    g = ConfigSpaceGrid(shape, [0, 0, 0], shape, cell_size=1.0, precision=precision)
    pos = np.full((3, 3), 1.5)
    MassAssignor(g, 0).add_particles(pos)
    g.clear()
    assert not g.data.any()  # read after a clear
    MassAssignor(g, 0).add_particles(pos)
    assert g.data[1, 1, 1] == 3.0
    MassAssignor(g, 0).add_particles(pos)
    view = g.data
    g.clear()
    assert not view.any()  # a held view sees it at once
    view[0, 0, 0] = 2.0
    assert g.sum() == 2.0  # and its writes are picked up
    del view
    MassAssignor(g, 0).add_particles(pos)
    g.clear()
    g += 0.1  # in double, whatever the device stores
    assert g.data[2, 3, 1] == 0.1
    g.clear()
    MassAssignor(g, 0).add_particles(pos)
    assert g.data.sum() == 3.0 and g.sum() == 3.0
