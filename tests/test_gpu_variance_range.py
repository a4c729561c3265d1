"""Variances at the ends of the floating range: sums of the elements that
would leave the type, squares that would, squares that would vanish, and means
far above the spread, in every length class of the row kernels (registers,
streamed; whole, ragged; the shortest rows), against float64 on the CPU."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

NAMES = {O.F32: "float32", O.BF16: "bfloat16", O.F16: "float16", O.F64: "float64"}
LOWEST = {O.F32: -np.finfo(np.float32).max, O.BF16: -3.3895313892515355e38, O.F16: -65504.0,
          O.F64: -np.finfo(np.float64).max}
# one chunk a lane, several, a block per row of four and eight waves, whole
# rows that fill their lanes, rows longer than registers hold
LENGTHS = [2, 5, 8, 37, 64, 256, 257, 512, 1000, 1024, 1027, 2048, 4095, 4096, 5000, 8192, 16384, 16387, 40000, 40001]


def _rows(dt, x):
    """x as a contiguous array and as the inside of a wider one (pitch n + 3, first column 1)."""
    from phptensors import CudaArray
    xs = O.to_storage(x.astype(np.float64 if dt == O.F64 else np.float32), dt)
    wide = np.zeros((x.shape[0], x.shape[1] + 3), xs.dtype)
    wide[:, 1:-2] = xs
    views = (CudaArray.fromNumpy(xs, NAMES[dt]), CudaArray.fromNumpy(wide, NAMES[dt]).slice(":", [1, x.shape[1] + 1]))
    return O.from_storage(xs, dt).astype(np.float64), views


@pytest.mark.parametrize("dt", list(NAMES), ids=NAMES.get)
@pytest.mark.parametrize("n", LENGTHS)
def test_rows_of_one_extreme_value(dt, n):
    lo = LOWEST[dt]
    x = np.stack([np.full(n, lo), np.full(n, -lo), np.full(n, lo)])
    for a in _rows(dt, x)[1]:
        assert a.var(1).toNumpy().tolist() == [0.0, 0.0, 0.0]
        assert a.std(1, 1).toNumpy().tolist() == [0.0, 0.0, 0.0]


@pytest.mark.parametrize("dt", [O.F32, O.BF16], ids=NAMES.get)
@pytest.mark.parametrize("n", LENGTHS)
def test_deviations_whose_squares_leave_float32(dt, n):
    """Masks beside ordinary values, values around 1e25 and around 1e-25: the
    standard deviation is a float32 where the variance is none."""
    from phptensors import synthetic
    z = synthetic.normal((3, n), 0.0, 1.0, seed=n).astype(np.float64)
    z[0, ::3] = LOWEST[dt]
    z[1] *= 1e25
    z[2] *= 1e-25
    x, views = _rows(dt, z)
    for a in views:
        got = a.std(1).toNumpy().astype(np.float64)
        # summed in double: at most n 2^-53 n of cancellation, then one rounding to float32
        assert np.allclose(got, x.std(1), rtol=2.0 ** -23, atol=0)


@pytest.mark.parametrize("n", LENGTHS)
def test_means_far_above_the_spread(n):
    """float32 rows of mean 1e5 and spread 1: the sums are double's, the result
    is rounded once."""
    from phptensors import synthetic
    x, views = _rows(O.F32, synthetic.normal((4, n), 1e5, 1.0, seed=n))
    for a in views:
        assert np.allclose(a.var(1).toNumpy().astype(np.float64), x.var(1), rtol=2.0 ** -23, atol=0)


@pytest.mark.parametrize("dt", [O.F32, O.BF16], ids=NAMES.get)
@pytest.mark.parametrize("n", [5, 37, 257, 1027, 4096, 5000, 40001])
def test_a_nonfinite_element_makes_the_variance_nan(dt, n):
    x = np.ones((6, n))
    x[0, 0], x[1, 0], x[2, n - 1], x[3, n // 2], x[4, n - 1] = np.inf, np.nan, -np.inf, np.inf, np.nan
    for a in _rows(dt, x)[1]:
        var = a.var(1).toNumpy()
        assert np.all(np.isnan(var[:5])) and var[5] == 0.0
