"""The eager elementwise kernels' 16-byte path (32- and 16-bit floats: flat,
unaligned, row-broadcast, column-broadcast and pitched operands, immediates)
against numpy, bit for bit: every operation used is correctly rounded in
float32 and then rounded to the type once.  Sizes around the 4 and 8 elements
of a chunk, rows that end inside chunks, and layouts the path refuses."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

NAMES = {O.F32: "float32", O.BF16: "bfloat16", O.F16: "float16"}
SHAPES = [(1, 1), (1, 7), (3, 3), (5, 8), (2, 9), (33, 31), (7, 1001), (260, 17), (64, 256), (1030, 5)]


def _values(shape, dt, seed):
    from phptensors import synthetic
    x = synthetic.normal(shape, 0.0, 2.0, seed=seed)
    x.reshape(-1)[::5] = np.round(x.reshape(-1)[::5])
    xs = O.to_storage(x, dt)
    return O.from_storage(xs, dt).astype(np.float32), xs


def _up(xs, dt):
    from phptensors import CudaArray
    return CudaArray.fromNumpy(xs, NAMES[dt])


def _layouts(shape, dt, seed):
    """(name, float32 values broadcast to shape, CudaArray) of one operand in every layout."""
    r, c = shape
    x, xs = _values(shape, dt, seed)
    yield "flat", x, _up(xs, dt)
    w = np.zeros((r, c + 3), xs.dtype)
    w[:, 1:c + 1] = xs
    yield "pitched", x, _up(w, dt).slice(":", [1, c + 1])
    f = np.zeros(r * c + 1, xs.dtype)
    f[1:] = xs.reshape(-1)
    yield "unaligned", x, _up(f, dt).slice([1, None]).reshape([r, c])
    yield "row", np.broadcast_to(x[:1], shape), _up(xs[:1].copy(), dt)
    yield "column", np.broadcast_to(x[:, :1], shape), _up(xs[:, :1].copy(), dt)
    yield "one", np.broadcast_to(x[:1, :1], shape), _up(xs[:1, :1].copy(), dt)
    yield "transposed", x, _up(np.ascontiguousarray(xs.T), dt).transpose()


def _same(got, ref, dt):
    """Bit for bit in the result's own type (float32 for 16-bit quotients); NaNs as NaNs."""
    if got.getDtype() == "float32":
        dt = O.F32
    bits = O.to_storage(np.asarray(ref, np.float32), dt)
    g = got.toBits()
    assert g.shape == bits.shape
    gf, rf = O.from_storage(g, dt), O.from_storage(bits, dt)
    ok = (g.view(bits.dtype) == bits) | (np.isnan(gf) & np.isnan(rf))
    assert np.all(ok), np.argwhere(~ok)[:3]


OPS = {"add": lambda a, b: a + b, "subtract": lambda a, b: a - b, "multiply": lambda a, b: a * b,
       "divide": lambda a, b: a / b, "maximum": lambda a, b: np.where(a > b, a, b),
       "minimum": lambda a, b: np.where(a < b, a, b), "gt": lambda a, b: (a > b).astype(np.float32),
       "eq": lambda a, b: (a == b).astype(np.float32), "le": lambda a, b: (a <= b).astype(np.float32)}


@pytest.mark.parametrize("dt", list(NAMES), ids=NAMES.get)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_binary_layouts(dt, shape):
    with np.errstate(all="ignore"):
        names = list(OPS)
        for i, (na, a, ca) in enumerate(_layouts(shape, dt, 1)):
            for j, (nb, b, cb) in enumerate(_layouts(shape, dt, 2)):
                full = np.broadcast_shapes(tuple(ca.getShape()), tuple(cb.getShape()))
                op = names[(i * 7 + j) % len(names)]
                ref = OPS[op](a, b).astype(np.float32)[:full[0], :full[1]]
                _same(getattr(ca, op)(cb), ref, dt)


@pytest.mark.parametrize("dt", list(NAMES), ids=NAMES.get)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_scalars_unary_and_casts(dt, shape):
    with np.errstate(all="ignore"):
        for name, a, ca in _layouts(shape, dt, 3):
            a = a[:ca.getShape()[0], :ca.getShape()[1]]
            _same(ca * 0.5, a * np.float32(0.5), dt)
            _same(0.5 - ca, np.float32(0.5) - a, dt)
            _same(ca.gt(0), (a > 0).astype(np.float32), dt)
            _same(ca.neg(), -a, dt)
            _same(ca.abs(), np.where(a < 0, -a, a), dt)
            _same(ca.floor(), np.floor(a), dt)
            _same(ca.abs().sqrt(), np.sqrt(np.where(a < 0, -a, a)), dt)
            _same(ca.astype("float32"), a, O.F32)


@pytest.mark.parametrize("dt", [O.BF16, O.F16], ids=NAMES.get)
@pytest.mark.parametrize("n", [1, 7, 8, 9, 1003])
def test_narrowing_casts(dt, n):
    """pt_cast from float32 (CudaArray.astype only widens), NaN and infinities included."""
    from phptensors import _abi as A
    x, xs = _values((n,), O.F32, n)
    x[0] = np.nan if n > 1 else x[0]
    x[-1] = np.inf if n > 8 else x[-1]
    src, dst = A.to_device(x), A.DeviceBuffer(2 * n)
    A.check(A.load().pt_cast(src.ptr, O.F32, A.sizes([1]), 0, dst.ptr, dt, A.ints([n]), 1, None))
    assert np.array_equal(dst.download(np.uint16, (n,)), O.to_storage(x, dt))


@pytest.mark.parametrize("dt", list(NAMES), ids=NAMES.get)
@pytest.mark.parametrize("cond", ["same", "bool", "int16", "int32", "int64", "float32"])
@pytest.mark.parametrize("shape", SHAPES[::2], ids=str)
def test_where_layouts(dt, cond, shape):
    from phptensors import CudaArray
    rng = np.random.default_rng(5)
    for i, (na, a, ca) in enumerate(_layouts(shape, dt, 6)):
        for j, (nb, b, cb) in enumerate(_layouts(shape, dt, 7)):
            if (i + j) % 3:
                continue
            pick = rng.integers(0, 2, shape)
            if cond == "same":
                vals = np.where(pick, 1.5, np.where(rng.integers(0, 2, shape), -0.0, 0.0)).astype(np.float32)
                vals.reshape(-1)[0], pick.reshape(-1)[0] = np.nan, 1  # NaN is unequal to zero
                cc = _up(O.to_storage(vals, dt), dt)
            else:
                cc = CudaArray.fromNumpy((pick * 3).astype(np.bool_ if cond == "bool" else cond), cond)
            _same(CudaArray.where(cc, ca, cb), np.where(pick, a, b), dt)
            got = CudaArray.where(cc.slice([0, 1]), ca, cb)  # one row of the condition for all
            _same(got, np.where(pick[:1], a, b)[:got.getShape()[0], :got.getShape()[1]], dt)


@pytest.mark.parametrize("dt", list(NAMES), ids=NAMES.get)
def test_three_dimensions_and_empty(dt):
    """A broadcast that does not collapse to rows keeps the general path; empty tensors launch nothing."""
    x, xs = _values((4, 5, 9), dt, 8)
    b, bs = _values((4, 1, 9), dt, 9)
    _same(_up(xs, dt) + _up(bs, dt), x + b, dt)
    e = _up(xs[:0], dt)
    assert (e + 1.0).getShape() == [0, 5, 9] and e.tanh().getShape() == [0, 5, 9]


@pytest.mark.parametrize("dt", list(NAMES), ids=NAMES.get)
def test_calls_past_the_caches(dt):
    """Tensors of 290 MB, an odd number of elements: the nontemporal forms give
    the bits of the cached ones (which short rows of the same values run)."""
    from phptensors import CudaArray
    rows, cols = (18311, 4097) if dt == O.F32 else (36601, 4099)
    _, a = _values((1, cols), dt, 10)
    _, b = _values((1, cols), dt, 11)
    tall = lambda s: _up(np.repeat(s, rows, 0), dt)
    x, m, x1, m1 = tall(a), tall(b), _up(a, dt), _up(b, dt)
    c, c1 = CudaArray.full([rows, 1], 1.25, NAMES[dt]), CudaArray.full([1, 1], 1.25, NAMES[dt])
    for name, big, small in (("pair", x + m, x1 + m1), ("scalar", x * 0.5, x1 * 0.5), ("reverse", 0.5 - x, 0.5 - x1),
                             ("row", x - m1, x1 - m1), ("row first", m1 - x, m1 - x1), ("column", x * c, x1 * c1),
                             ("column first", c - x, c1 - x1), ("unary", x.neg(), x1.neg()), ("quotient", x / m, x1 / m1),
                             ("tanh", x.tanh(), x1.tanh()), ("where", CudaArray.where(x.gt(0), x, m),
                                                              CudaArray.where(x1.gt(0), x1, m1))):
        got, ref = big.toBits(), small.toBits()
        assert got.shape == (rows, cols) and got.dtype == ref.dtype, name
        assert np.array_equal(got.view(np.uint8), np.broadcast_to(ref, (rows, cols)).copy().view(np.uint8)), name
        del big, got
