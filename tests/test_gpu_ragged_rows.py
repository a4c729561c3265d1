"""GPU parity of the last-axis kernels on rows whose length, pitch or base is
no multiple of 16 bytes: reductions, softmax and layerNorm read them in
16-byte chunks at any element, with one lane straddling the row's end.
Lengths around the chunk and wave counts where the kernels change, against
float64 on the CPU."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

NAMES = {O.F32: "float32", O.BF16: "bfloat16", O.F16: "float16", O.F64: "float64"}
LENGTHS = [1, 3, 9, 63, 129, 255, 257, 511, 513, 1001, 1023, 1025, 2047, 2049, 4095, 4097, 8191, 8193, 16383, 16385,
           33001]


def _arrays(dt, n, seed):
    """[5, n] values as a contiguous array and as the inside of a wider one (pitch n + 3, first column 1)."""
    from phptensors import CudaArray, synthetic
    x = synthetic.normal((5, n), 0.25, 1.0, seed=seed)
    x[1] = np.round(x[1] * 2) / 2          # ties
    x[2, n // 2:] = x[2, n // 2]
    xs = O.to_storage(x.astype(np.float64) if dt == O.F64 else x, dt)
    wide = np.zeros((5, n + 3), xs.dtype)
    wide[:, 1:n + 1] = xs
    whole = CudaArray.fromNumpy(xs, NAMES[dt])
    view = CudaArray.fromNumpy(wide, NAMES[dt]).slice(":", [1, n + 1])
    return O.from_storage(xs, dt).astype(np.float64), whole, view


@pytest.mark.parametrize("dt", list(NAMES), ids=NAMES.get)
@pytest.mark.parametrize("n", LENGTHS)
def test_ragged_rows(dt, n):
    x, whole, view = _arrays(dt, n, n)
    # float32 sums of n terms in any order: n 2^-24 sum|x| covers it (n 2^-53 in float64)
    u = 2.0 ** -53 if dt == O.F64 else 2.0 ** -24
    bound = n * u * np.abs(x).sum(1) + 1e-300
    for a in (whole, view):
        assert np.all(np.abs(a.sum(1).toNumpy().astype(np.float64) - x.sum(1)) <= bound)
        assert np.array_equal(a.max(1).toNumpy().astype(np.float64), x.max(1))
        assert np.array_equal(a.min(1).toNumpy().astype(np.float64), x.min(1))
        assert np.array_equal(a.argMax(1).toNumpy(), x.argmax(1))
        assert np.array_equal(a.argMin(1).toNumpy(), x.argmin(1))
        var = a.var(1).toNumpy().astype(np.float64)
        # two passes or Welford over n terms; the row's spread is of the order of its values
        assert np.allclose(var, x.var(1), rtol=32 * u * max(n, 8) ** 0.5, atol=1e-30)


@pytest.mark.parametrize("dt", list(NAMES), ids=NAMES.get)
@pytest.mark.parametrize("rows", [1023, 1026])
@pytest.mark.parametrize("n", [321, 353, 801, 1025, 2049, 4095, 4099, 8191])
def test_ragged_rows_of_a_full_grid(dt, rows, n):
    """Where the rows alone fill the chip, up to 16 chunks take a wave each; a
    block of four of them ends past the last row."""
    from phptensors import CudaArray, synthetic
    x = synthetic.normal((rows, n), 0.25, 1.0, seed=n)
    x[1] = np.round(x[1] * 2) / 2
    xs = O.to_storage(x.astype(np.float64) if dt == O.F64 else x, dt)
    a, x = CudaArray.fromNumpy(xs, NAMES[dt]), O.from_storage(xs, dt).astype(np.float64)
    u = 2.0 ** -53 if dt == O.F64 else 2.0 ** -24  # bounds as above
    assert np.all(np.abs(a.sum(1).toNumpy().astype(np.float64) - x.sum(1)) <= n * u * np.abs(x).sum(1))
    assert np.array_equal(a.max(1).toNumpy().astype(np.float64), x.max(1))
    assert np.array_equal(a.argMax(1).toNumpy(), x.argmax(1))
    assert np.array_equal(a.argMin(1).toNumpy(), x.argmin(1))
    assert np.allclose(a.var(1).toNumpy().astype(np.float64), x.var(1), rtol=32 * u * n ** 0.5, atol=0)


@pytest.mark.parametrize("dt", list(NAMES), ids=NAMES.get)
@pytest.mark.parametrize("n", LENGTHS)
def test_ragged_softmax_and_layernorm(dt, n):
    x, whole, view = _arrays(dt, n, n + 7)
    _check_normalized(dt, n, x, (whole, view))


@pytest.mark.parametrize("rows", [1023, 1024, 1026])
@pytest.mark.parametrize("n", [1025, 1281, 1534, 2047])
def test_ragged_normalization_of_a_full_grid(rows, n):
    """fp32 rows that take a wave each, and those one row short of it."""
    from phptensors import CudaArray, synthetic
    x = synthetic.normal((rows, n), 0.25, 1.0, seed=n)
    _check_normalized(O.F32, n, x.astype(np.float64), (CudaArray.fromNumpy(x),))
    x[0, n - 1], x[1, 0], x[2] = np.nan, np.inf, -np.inf
    bad = CudaArray.fromNumpy(x)
    for got in (bad.softmax(1).toNumpy(), bad.layerNorm([1], 1e-5).toNumpy()):
        assert np.all(np.isnan(got[:3]).any(1)) and np.all(np.isfinite(got[3:]))


def _check_normalized(dt, n, x, arrays):
    from phptensors import CudaArray, synthetic
    u = 2.0 ** -53 if dt == O.F64 else 2.0 ** -24
    e = np.exp(x - x.max(1, keepdims=True))
    soft = e / e.sum(1, keepdims=True)
    g = synthetic.normal((n,), 1.0, 0.1, seed=3)
    b = synthetic.normal((n,), 0.0, 0.1, seed=4)
    pdt = "float64" if dt == O.F64 else "float32"
    ga, ba = CudaArray.fromNumpy(g.astype(pdt), pdt), CudaArray.fromNumpy(b.astype(pdt), pdt)
    norm = (x - x.mean(1, keepdims=True)) / np.sqrt(x.var(1, keepdims=True) + 1e-5)
    for a in arrays:
        # expf to 2 ulp, the sum's and the quotient's rounding
        got = a.softmax(1).toNumpy().astype(np.float64)
        assert np.allclose(got, soft, rtol=(16 + n ** 0.5) * u, atol=1e-30)
        # the mean's error (sqrt(n) u of values of order 1) over the deviation, which is of order 1 or sqrt(eps)
        scale = 1.0 / np.sqrt(x.var(1, keepdims=True) + 1e-5)
        tol = (16 + n ** 0.5) * u * (1.0 + np.abs(norm) + scale) * 2
        got = a.layerNorm([1], 1e-5, ga, ba).toNumpy().astype(np.float64)
        assert np.all(np.abs(got - (norm * g + b)) <= tol * 1.5)
        got = a.layerNorm([1], 1e-5).toNumpy().astype(np.float64)
        assert np.all(np.abs(got - norm) <= tol)


def test_ragged_nonfinite_rows():
    """NaN and infinities in the straddling lane's elements."""
    from phptensors import CudaArray
    for n in (261, 1029, 4097):
        x = np.ones((6, n), np.float32)
        x[0, n - 1], x[1, n - 1], x[2, n - 1] = np.nan, np.inf, -np.inf
        x[3] = -np.inf
        x[4, 0] = np.nan
        a = CudaArray.fromNumpy(x)
        assert a.argMax(1).toNumpy().tolist() == [0, n - 1, 0, 0, 1, 0]
        assert a.max(1).toNumpy().tolist() == [1.0, np.inf, 1.0, -np.inf, 1.0, 1.0]
        var = a.var(1).toNumpy()
        assert np.all(np.isnan(var[:5])) and var[5] == 0.0
        soft = a.softmax(1).toNumpy()
        assert np.all(np.isnan(soft[[0, 1, 3, 4]][:, 0])) and np.all(np.isfinite(soft[[2, 5]]))
        assert soft[2, n - 1] == 0.0


@pytest.mark.parametrize("dt", ["bfloat16", "float16"])
@pytest.mark.parametrize("n", [1, 7, 8, 512, 1001, 4096, 16385, 40000])
def test_layernorm_parameters_of_the_inputs_type(dt, n):
    """Scale and bias in the input's 16-bit type give the bits that their
    widened values give, together or alone; mixed types still cast."""
    from phptensors import CudaArray, synthetic
    code = {"bfloat16": O.BF16, "float16": O.F16}[dt]
    up = lambda v: CudaArray.fromNumpy(O.to_storage(v, code), dt)  # noqa: E731
    x = up(synthetic.normal((4, n), 0.5, 2.0, seed=n))
    g, b = up(synthetic.normal((n,), 1.0, 0.2, seed=1)), up(synthetic.normal((n,), 0.0, 0.2, seed=2))
    gf, bf = g.astype("float32"), b.astype("float32")
    bits = lambda s, t: x.layerNorm([1], 1e-5, s, t).toBits().view(np.uint32)  # noqa: E731
    ref = bits(gf, bf)
    assert np.array_equal(bits(g, b), ref) and np.array_equal(bits(g, bf), ref)
    assert np.array_equal(bits(g, None), bits(gf, None)) and np.array_equal(bits(None, b), bits(None, bf))
