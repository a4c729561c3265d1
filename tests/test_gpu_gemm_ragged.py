"""GPU parity of the products at sizes that fill no whole tiles, K steps or
16-byte packs: integer-valued operands, so that every order of summation gives
the same bits, against the float64 product; every operand layout, contiguous
and inside wider arrays, with NaN in the memory that a tail must not use."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

NAMES = {O.F32: "float32", O.BF16: "bfloat16", O.F16: "float16"}


def _operand(shape, dt, transposed, wide, seed):
    """Integer values [-4, 4] and a CudaArray of them: row-major or transposed in memory, contiguous or
    surrounded by NaN."""
    from phptensors import CudaArray, synthetic
    x = synthetic.integers(shape, -4, 5, seed=seed).astype(np.float32)
    m = np.ascontiguousarray(np.swapaxes(x, -1, -2)) if transposed else x
    if wide:
        pad = wide
        w = np.full(m.shape[:-2] + (m.shape[-2] + 2, m.shape[-1] + pad), np.nan, np.float32)
        w[..., 1:-1, pad - 1:pad - 1 + m.shape[-1]] = m
        a = CudaArray.fromNumpy(O.to_storage(w, dt), NAMES[dt])
        a = a.slice(*([":"] * (m.ndim - 2)), [1, m.shape[-2] + 1], [pad - 1, pad - 1 + m.shape[-1]])
    else:
        a = CudaArray.fromNumpy(O.to_storage(m, dt), NAMES[dt])
    return x, a.swapaxes(-1, -2) if transposed else a


def _check(dt, bmnk, ta, tb, wide):
    b, m, n, k = bmnk
    x, a = _operand((b, m, k), dt, ta, wide, m + k)
    y, c = _operand((b, k, n), dt, tb, wide, n + k)
    got = a.matmul(c).toBits()
    ref = np.matmul(x.astype(np.float64), y.astype(np.float64)).astype(np.float32)
    assert np.array_equal(got.view(np.float32) if dt == O.F32 else got, O.to_storage(ref, dt))


@pytest.mark.parametrize("ta", [False, True], ids=["A", "At"])
@pytest.mark.parametrize("tb", [False, True], ids=["B", "Bt"])
@pytest.mark.parametrize("k", [1, 2, 4, 8, 12, 20, 31, 33, 36, 100, 127, 1000, 1004])
def test_fp32_k_tails(ta, tb, k):
    """The ring kernel's last step at every kind of remainder, whole and split K."""
    for b, m, n in ((1, 128, 128), (2, 260, 132), (1, 256, 384)):
        _check(O.F32, (b, m, n, k), ta, tb, 0)
    _check(O.F32, (1, 128, 132, 4 * k + 2048), ta, tb, 0)
    _check(O.F32, (1, 128, 128, k), ta, tb, 4)


@pytest.mark.parametrize("dt", list(NAMES), ids=NAMES.get)
@pytest.mark.parametrize("ta", [False, True], ids=["A", "At"])
@pytest.mark.parametrize("tb", [False, True], ids=["B", "Bt"])
@pytest.mark.parametrize("mnk", [(1, 1, 1), (17, 33, 5), (64, 64, 32), (65, 63, 33), (127, 129, 31), (129, 127, 65),
                                 (130, 131, 96), (131, 257, 100), (255, 130, 777), (257, 383, 40), (300, 301, 302)],
                         ids=str)
def test_ragged_products(dt, ta, tb, mnk):
    for wide in (0, 1, 3):
        _check(dt, (1,) + mnk, ta, tb, wide)
    _check(dt, (3,) + mnk, ta, tb, 1)


@pytest.mark.parametrize("dt", list(NAMES), ids=NAMES.get)
@pytest.mark.parametrize("ta", [False, True], ids=["A", "At"])
@pytest.mark.parametrize("tb", [False, True], ids=["B", "Bt"])
def test_ragged_split_k_and_large_tiles(dt, ta, tb):
    _check(dt, (1, 131, 70, 2999), ta, tb, 0)   # split K
    _check(dt, (1, 65, 257, 4097), ta, tb, 1)
    _check(dt, (9, 1300, 1291, 70), ta, tb, 0)  # 256x256 tiles


@pytest.mark.parametrize("dt", list(NAMES), ids=NAMES.get)
def test_nonfinite_operands_stay_in_their_rows(dt):
    """Infinities and NaN next to a K tail reach exactly the outputs whose sums hold them."""
    from phptensors import CudaArray, synthetic
    m, n, k = 131, 133, 69
    x = synthetic.integers((m, k), 1, 5, seed=1).astype(np.float32)
    y = synthetic.integers((k, n), 1, 5, seed=2).astype(np.float32)
    x[5, k - 1], x[6, 0], y[k - 1, 7], y[40, 9] = np.inf, np.nan, -np.inf, np.nan
    for tb in (False, True):
        c = CudaArray.fromNumpy(O.to_storage(np.ascontiguousarray(y.T) if tb else y, dt), NAMES[dt])
        got = CudaArray.fromNumpy(O.to_storage(x, dt), NAMES[dt]).matmul(c.T if tb else c).toNumpy()
        ref = x.astype(np.float64) @ y.astype(np.float64)
        assert np.array_equal(np.isnan(got), np.isnan(ref))
        assert np.array_equal(np.isinf(got), np.isinf(ref))
        f = np.isfinite(ref)
        assert np.array_equal(got[f].astype(np.float32),
                              O.from_storage(O.to_storage(ref[f].astype(np.float32), dt), dt).astype(np.float32))
