"""GPU parity of the products at sizes that fill no whole tiles, K steps or
16-byte packs: integer-valued operands, so that every order of summation gives
the same bits, against the float64 product; every operand layout, contiguous
and inside wider arrays, with NaN in the memory that a tail must not use: rows
at any element (the register-staged kernels) and aligned ones (the fp32 ring)."""
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
    """The last K step at every kind of remainder, whole and split K."""
    for b, m, n in ((1, 128, 128), (2, 260, 132), (1, 256, 384)):
        _check(O.F32, (b, m, n, k), ta, tb, 0)
    _check(O.F32, (1, 128, 132, 4 * k + 2048), ta, tb, 0)
    _check(O.F32, (1, 128, 128, k), ta, tb, 4)


def _padded(shape, transposed, before, seed):
    """Integer values inside an array whose pitch is the next multiple of 4
    after `before` + the row, at column `before` (0 or 4: packs stay aligned),
    NaN in every other element; the array ends with the last row's last
    element.  Returns the values and the array's memory, base, pitch."""
    from phptensors import synthetic
    x = synthetic.integers(shape, -4, 5, seed=seed).astype(np.float32)
    m = np.ascontiguousarray(x.T) if transposed else x
    pitch = (before + m.shape[1] + 4) // 4 * 4
    w = np.full((m.shape[0], pitch), np.nan, np.float32)
    w[:, before:before + m.shape[1]] = m
    return x, w.ravel()[:(m.shape[0] - 1) * pitch + before + m.shape[1]], before, pitch


@pytest.mark.parametrize("ta", [False, True], ids=["A", "At"])
@pytest.mark.parametrize("tb", [False, True], ids=["B", "Bt"])
@pytest.mark.parametrize("before", [0, 4])
@pytest.mark.parametrize("k", [2, 3, 5, 29, 30, 31, 33, 63, 69, 98, 125, 126, 127])
def test_fp32_ring_beside_nan(ta, tb, before, k):
    """The ring kernel's K tail in operands of aligned, padded rows: every
    remainder of K, in a k-contiguous operand the last pack straddles the end
    of K (and of the array in the last row), and what lies past K is NaN."""
    from phptensors import _abi as A
    lib = A.load()
    A.check(lib.pt_init(), "init")
    for m, n in ((128, 128), (132, 260)):
        x, xm, xo, xp = _padded((m, k), ta, before, m + k)
        y, ym, yo, yp = _padded((k, n), tb, before, n + k)
        da, db, dc = A.to_device(xm), A.to_device(ym), A.DeviceBuffer(4 * m * n)
        for tile in (38, -1):  # the ring, and what the dispatch takes for so short a K
            A.check(lib.pt_matmul_set_tile(tile))
            try:
                A.matmul(da.ptr + 4 * xo, db.ptr + 4 * yo, dc.ptr, A.FLOAT32, (m, k), [1, xp] if ta else [xp, 1],
                         (k, n), [1, yp] if tb else [yp, 1], (m, n))
            finally:
                lib.pt_matmul_set_tile(-1)
            assert (A.backend_info().last_matmul.decode() == "mfma-fp32-ring") == (tile == 38)
            assert np.array_equal(dc.download(np.float32, (m, n)), (x.astype(np.float64) @ y.astype(np.float64)))


@pytest.mark.parametrize("k", [383, 385, 777, 1002])
def test_fp32_ring_beside_nan_on_a_full_grid(k):
    """The same where the tiles alone fill the CUs, as columns of wider tensors."""
    from phptensors import CudaArray, _abi, synthetic
    m, n = 2052, 2050
    x = synthetic.integers((m, k), -4, 5, seed=1).astype(np.float32)
    y = synthetic.integers((n, k), -4, 5, seed=2).astype(np.float32)
    wide = []
    for v in (x, y):
        w = np.full((v.shape[0], 1008), np.nan, np.float32)
        w[:, 4:4 + k] = v
        wide.append(CudaArray.fromNumpy(w).slice(":", [4, 4 + k]))
    got = wide[0].matmul(wide[1].T).toNumpy()
    assert (_abi.backend_info().last_matmul.decode() == "mfma-fp32-ring") == (k >= 384)
    assert np.array_equal(got, x.astype(np.float64) @ y.astype(np.float64).T)


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


@pytest.mark.parametrize("dt", [O.BF16, O.F16], ids=NAMES.get)
@pytest.mark.parametrize("ta", [False, True], ids=["A", "At"])
@pytest.mark.parametrize("tb", [False, True], ids=["B", "Bt"])
@pytest.mark.parametrize("bmn,ks", [((1, 510, 1024), (2048, 2050)), ((1, 1150, 2046), (640, 641, 1024, 1025)),
                                    ((2, 900, 1500), (640, 641, 896, 897, 1024)), ((1, 2048, 2046), (1024, 1025)),
                                    ((5, 900, 850), (64, 65, 128, 129)), ((13, 900, 850), (128, 129, 512, 513))],
                         ids=str)
def test_both_sides_of_the_16_bit_tile_rule(dt, ta, tb, bmn, ks):
    """64x64 tiles, 128x128 tiles with K split, of four waves and of eight, by number of tiles, K and layout."""
    for k in ks:
        _check(dt, bmn + (k,), ta, tb, 0)


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
