"""Mixed-radix row passes stay within 64 KB of LDS a workgroup at every length
they take (host arithmetic of the plan, no GPU)."""
import ctypes

import pytest

from fftcorr_amd import _lib


def row_lds(n2, precision):
    b = ctypes.c_size_t()
    _lib.check(_lib.lib().fc_fft_row_lds(n2, _lib.precision_code(precision), ctypes.byref(b)))
    return b.value


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_rows_stay_within_64_kb(precision):
    over = [(n, row_lds(n, precision)) for n in range(1, 4097)
            if row_lds(n, precision) > 65536]
    assert not over, (len(over), over[:5])


def test_which_lengths_take_the_stages():
    assert row_lds(512, "fp64") == 0 and row_lds(384, "fp32") == 0  # compile-time plans
    assert row_lds(4093, "fp64") == 0  # prime, too long for a chirp convolution: direct sums
    # One row of n values and a gap after every eighth, in FP64.
    assert row_lds(3600, "fp64") == 16 * (3600 + 450 + 1)
    assert row_lds(400, "fp64") > 0 and row_lds(1999, "fp32") > 32768
