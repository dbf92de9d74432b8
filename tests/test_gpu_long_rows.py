"""Row passes of long rows without a compile-time plan (csrc/fft_gen_rows.hip):
the lengths whose LDS row leaves room for fewer gaps than the short ones, or for
none (chirp convolutions over 4096 points), against numpy.  Tolerances as
tests/test_gpu_fft.py: FP64 1e-12 log2(N), FP32 3e-6 log2(N) of the largest
value."""
import numpy as np
import pytest

from gpu_helpers import fft_c2r, fft_r2c

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-12, "fp32": 3e-6}


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n2", [1801, 1820, 1999, 2047, 3600, 3645, 3780, 3888, 3969, 4000, 4050])
@pytest.mark.parametrize("rows", [(2, 2), (1, 3)])
def test_transforms_match_numpy(rows, n2, precision):
    shape = rows + (n2,)
    rng = np.random.default_rng(n2 + rows[1])
    a = rng.normal(size=shape)
    tol = TOL[precision] * np.log2(a.size)
    ref = np.fft.rfftn(a)
    assert np.max(np.abs(fft_r2c(a, precision) - ref)) <= tol * np.max(np.abs(ref))
    back = np.fft.irfftn(ref, s=shape, axes=(0, 1, 2), norm="forward")
    assert np.max(np.abs(fft_c2r(ref, shape, precision) - back)) <= tol * np.max(np.abs(back))
