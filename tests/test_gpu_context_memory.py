"""What a context keeps: page-locked staging only from the first host catalogue
that is copied through it (4 MB and more), all of it given back on request."""
import ctypes

import numpy as np
import pytest

from fftcorr_amd import _lib

pytestmark = pytest.mark.gpu

SMALL, LARGE = 1 << 20, 16 << 20  # results; the staging slots


def host_bytes(ctx):
    b = ctypes.c_size_t()
    _lib.check(_lib.lib().fc_ctx_host_footprint(ctx.handle, ctypes.byref(b)))
    return b.value


def assign(grid, n):
    pos = np.random.default_rng(n).uniform(0, 8, (n, 3))
    st = _lib.MaStats()
    _lib.check(_lib.lib().fc_mass_assign(grid.handle, _lib.dptr(pos), n, 3, None, 1.0, 0, 1, 0.0,
                                         ctypes.byref(st)))
    assert st.num_added == n and st.totw == n


def test_staging_memory_comes_with_the_first_large_catalogue():
    ctx = _lib.Context(0)
    grid = _lib.DeviceGrid((8, 8, 8), cell_size=1.0, ctx=ctx)
    assert host_bytes(ctx) == 0
    assign(grid, 1000)
    assign(grid, (4 << 20) // 24)
    assert 0 < host_bytes(ctx) < SMALL
    assign(grid, (4 << 20) // 24 + 1)
    assert LARGE <= host_bytes(ctx) < LARGE + SMALL
    _lib.check(_lib.lib().fc_ctx_release_scratch(ctx.handle))
    assert host_bytes(ctx) == 0
    held = ctypes.c_size_t()
    _lib.check(_lib.lib().fc_ctx_footprint(ctx.handle, ctypes.byref(held)))
    assert held.value == 0
    assign(grid, 300_000)
    total = 1000 + (4 << 20) // 24 * 2 + 1 + 300_000
    assert grid.stats()[0] == total
