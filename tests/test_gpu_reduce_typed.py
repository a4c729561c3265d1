"""GPU parity of the typed reductions over non-last axes and over all
elements: argmax / argmin / variance along columns and every op over a whole
tensor, at the edges of their blocks (columns per block, a straddling last
lane, one and several row slices, whole and partial chunks, one and several
blocks), against the CPU oracle."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

DTS = [O.F32, O.F64, O.BF16, O.F16]
NAMES = {O.F32: "f32", O.F64: "f64", O.BF16: "bf16", O.F16: "f16"}


@pytest.fixture(scope="module")
def G():
    import gpu_util
    from phptensors import _abi
    _abi.load()
    _abi.check(_abi.load().pt_init(), "init")
    return gpu_util


def _ints(shape, dt, seed):
    """Small whole numbers: every sum exact, many ties."""
    from phptensors import synthetic
    x = np.round(synthetic.uniform(shape, -40.0, 40.0, seed=seed)).astype(np.float32)
    return x, O.to_storage(x.astype(np.float64) if dt == O.F64 else x, dt)


def _check_var(G, xs, dt, axis):
    """float64: Welford's updates, a few roundings of 2^-53 a term that add up
    like sqrt(n).  The others are summed in double and rounded to float32 once."""
    x = O.from_storage(xs, dt).astype(np.float64)
    # numpy adds a contiguous last axis pairwise, any other one element after
    # element (3e-13 off the exact variance of 20000 whole numbers)
    x = x.ravel() if axis is None else np.ascontiguousarray(np.moveaxis(x, axis, -1))
    n = x.shape[-1]
    rtol = 16 * 2.0 ** -53 * max(n, 16) ** 0.5 if dt == O.F64 else 2.0 ** -23
    for corr, std in ((0, False), (1, True)):
        if n <= corr:
            continue
        got = np.asarray(G.moments(xs, dt, axis, corr, std), np.float64).ravel()
        ref = np.atleast_1d(x.std(-1, ddof=corr) if std else x.var(-1, ddof=corr)).ravel()
        assert np.allclose(got, ref, rtol=rtol, atol=0, equal_nan=True), (corr, std)


@pytest.mark.parametrize("dt", DTS, ids=NAMES.get)
@pytest.mark.parametrize("shape,axis", [((2, 3), 0), ((3, 5, 1), 1), ((130, 31), 0), ((257, 129), 0), ((64, 257), 0),
                                        ((4097, 1001), 0), ((5, 70, 513), 1), ((20000, 40), 0), ((70, 33000), 0)],
                         ids=str)
def test_column_arg_and_variance(G, dt, shape, axis):
    x, xs = _ints(shape, dt, 11 + shape[0])
    for op in ("argmax", "argmin"):
        assert np.array_equal(G.arg_reduce(xs, dt, op, axis), O.arg_reduce(xs, dt, op, axis)), op
    _check_var(G, xs, dt, axis)
    for op in ("sum", "max"):
        got, _ = G.reduce(xs, dt, op, axis)
        assert np.array_equal(got, O.reduce(xs, dt, op, axis)[0]), op


@pytest.mark.parametrize("dt", DTS, ids=NAMES.get)
@pytest.mark.parametrize("n", [1, 7, 255, 1024, 4096, 4097, 16385, 300001])
def test_global_reductions(G, dt, n):
    x, xs = _ints((n,), dt, n)
    for op in ("argmax", "argmin"):
        assert np.array_equal(G.arg_reduce(xs, dt, op, None), O.arg_reduce(xs, dt, op, None)), op
    for op in ("sum", "max", "min"):
        got, rdt = G.reduce(xs, dt, op, None)
        ref, rrdt = O.reduce(xs, dt, op, None)
        assert rdt == rrdt and np.array_equal(got.ravel(), ref.ravel()), op
    got, _ = G.reduce(xs, dt, "mean", None)
    assert np.allclose(got.ravel(), O.reduce(xs, dt, "mean", None)[0].ravel(), rtol=2e-7, atol=0)
    _check_var(G, xs, dt, None)


@pytest.mark.parametrize("dt", DTS, ids=NAMES.get)
@pytest.mark.parametrize("axis", [0, None])
def test_nonfinite_values(G, dt, axis):
    """NaN is never taken by arg reductions, a column without any value above
    -inf (below inf) gives index 0, and NaN or an infinity anywhere makes a
    variance NaN."""
    x, _ = _ints((700, 140), dt, 5)
    x[3, 0] = x[0, 1] = np.nan
    x[:, 2], x[:, 3], x[:, 4] = -np.inf, np.inf, np.nan
    x[699, 5], x[0, 6] = np.inf, -np.inf
    x[:, 7], x[350, 7] = -np.inf, np.nan
    xs = O.to_storage(x.astype(np.float64) if dt == O.F64 else x, dt)
    for op in ("argmax", "argmin"):
        assert np.array_equal(G.arg_reduce(xs, dt, op, axis), O.arg_reduce(xs, dt, op, axis)), op
    got = np.asarray(G.moments(xs, dt, axis)).ravel()
    if axis is None:
        assert np.isnan(got[0])
    else:
        assert np.all(np.isnan(got[:8])) and np.all(np.isfinite(got[8:]))


@pytest.mark.parametrize("dt", DTS, ids=NAMES.get)
@pytest.mark.parametrize("shape", [(5003, 301), (9001, 1003)], ids=str)
def test_nonfinite_values_of_a_straddling_lane(G, dt, shape):
    """The same in the last columns, which the lane that straddles the row's
    end loads one by one, in the first, a middle and the last of several row
    slices."""
    x, _ = _ints(shape, dt, 6)
    last, mid = shape[0] - 1, shape[0] // 2
    x[mid, -1] = x[0, -2] = x[last, -3] = np.nan
    x[:, -4], x[:, -5], x[:, -6] = -np.inf, np.inf, np.nan
    x[last, -7], x[0, -8] = np.inf, -np.inf
    x[:, -9], x[mid, -9] = -np.inf, 3.0
    xs = O.to_storage(x.astype(np.float64) if dt == O.F64 else x, dt)
    for op in ("argmax", "argmin"):
        assert np.array_equal(G.arg_reduce(xs, dt, op, 0), O.arg_reduce(xs, dt, op, 0)), op
    for op in ("sum", "max", "min"):
        assert np.array_equal(G.reduce(xs, dt, op, 0)[0], O.reduce(xs, dt, op, 0)[0], equal_nan=True), op
    got = np.asarray(G.moments(xs, dt, 0)).ravel()
    assert np.all(np.isnan(got[-9:])) and np.all(np.isfinite(got[:-9]))


def test_variance_far_from_zero(G):
    """A mean far above the spread, and a first value far from the others."""
    from phptensors import synthetic
    x = synthetic.normal((5000, 70), 1e4, 1.0, seed=9).astype(np.float32)
    x[0, 10:20] = -3e4
    for axis in (0, None):
        _check_var(G, x, O.F32, axis)


@pytest.mark.parametrize("shape,axis", [((5000, 70), 0), ((70, 3, 50), 1), ((3, 5, 1), 1), ((257, 129), 0),
                                        ((200000, 40), 0), ((1100, 5000, 1), 1), ((9001,), None),
                                        ((4000003,), None)], ids=str)
def test_float64_variance_is_float64_accurate(G, shape, axis):
    """Ordinary values, and an outlier in first place (of every column, of the
    tensor): the error is a few roundings of the result, not of the outlier's
    square over the spread."""
    from phptensors import synthetic
    x = synthetic.normal(shape, 0.5, 1.0, seed=3).astype(np.float64)
    _check_var(G, x, O.F64, axis)
    x[0 if axis != 1 else (slice(None), 0)] = 1e6
    _check_var(G, x, O.F64, axis)


@pytest.mark.parametrize("axis", [0, None])
def test_float64_variance_at_the_ends_of_its_range(G, axis):
    """One extreme value everywhere has variance 0, finite values whose
    variance leaves float64 have variance inf."""
    for n in (3, 4, 17, 300, 5000):
        for v in (np.finfo(np.float64).max, -np.finfo(np.float64).max):
            assert np.all(np.asarray(G.moments(np.full((n, 5), v), O.F64, axis)) == 0.0)
        x = np.full((n, 5), 1e200)
        x[n // 2] = -1e200
        assert np.all(np.asarray(G.moments(x, O.F64, axis)) == np.inf)


def test_global_reduction_of_an_offset_view(G):
    """A base that is no multiple of 16 bytes."""
    x, xs = _ints((9001,), O.BF16, 3)
    for off in (1, 3, 8):
        from phptensors import CudaArray
        v = CudaArray.fromNumpy(xs, "bfloat16").slice([off, None])
        assert v.sum().item() == float(x[off:].sum())
        assert v.argMax().item() == int(np.argmax(x[off:]))


@pytest.mark.parametrize("shape", [(1000, 18075), (8000, 3001), (700, 66001)], ids=str)
@pytest.mark.parametrize("op", ["max", "min", "sum"])
def test_unaligned_columns_fit_the_static_scratch(shape, op):
    """Column reductions whose slices of 64-column blocks fit the megabyte of
    the no-allocation entry still fit it, with pt_reduce's bits."""
    from phptensors import _abi as A
    x = np.random.default_rng(4).integers(0, 0x3F80, shape, dtype=np.uint16)
    rows, cols = shape
    dx, one, two = A.to_device(x), A.DeviceBuffer(cols * 4), A.DeviceBuffer(cols * 4)
    lib = A.load()
    args = (A.BFLOAT16, A.OP[op], A.ints(shape), A.sizes([cols, 1]), 2, 0, 0, None)
    A.check(lib.pt_reduce_noalloc(dx.ptr, one.ptr, *args), "reduction without allocation")
    A.check(lib.pt_reduce(dx.ptr, two.ptr, *args), "reduction")
    got = one.download(np.float32, (cols,))
    assert np.array_equal(got, two.download(np.float32, (cols,)))
    if op != "sum":
        ref = O.from_storage(x, O.BF16).astype(np.float32)
        assert np.array_equal(got, ref.max(0) if op == "max" else ref.min(0))
