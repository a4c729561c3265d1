"""Row gathers by a broadcast index (16 bytes per thread, the last chunk moved
back to the row's end) and their validation, which looks at each index once:
row widths around a chunk, pitched tables, every element size, invalid
indices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["float64", "float32", "float16", "bfloat16", "int8"])
@pytest.mark.parametrize("width", [1, 2, 3, 4, 7, 8, 15, 16, 17, 33, 256, 1001])
@pytest.mark.parametrize("pitched", [False, True])
def test_rows(dt, width, pitched):
    from phptensors import CudaArray
    rng = np.random.default_rng(width)
    bits = {"float64": np.float64, "int8": np.int8}.get(dt, np.float32)
    t = rng.integers(-100, 100, (37, width + 5)).astype(bits)
    if dt in ("float16", "bfloat16"):
        t = rng.integers(0, 2 ** 15, t.shape).astype(np.uint16) & 0x3BFF
    table = CudaArray.fromNumpy(t if pitched else np.ascontiguousarray(t[:, 3:3 + width]), dt)
    if pitched:
        table = table.slice(":", [3, 3 + width])
    i = rng.integers(0, 37, (101, 1)).astype(np.int32)
    index = CudaArray.fromNumpy(i)
    got = table.gather(index.broadcastTo([101, width]), 0).toBits()
    ref = t[i[:, 0], 3:3 + width]
    assert np.array_equal(got.view(ref.dtype), ref)
    # the same through a whole index array, which the general kernel takes
    full = CudaArray.fromNumpy(np.ascontiguousarray(np.broadcast_to(i, (101, width))))
    assert np.array_equal(table.gather(full, 0).toBits(), got)


@pytest.mark.parametrize("bad", [-1, 37, 2 ** 31 - 1])
def test_invalid_index_is_found_in_a_broadcast(bad):
    from phptensors import CudaArray
    from phptensors._abi import InvalidArgumentException
    table = CudaArray.fromNumpy(np.ones((37, 64), np.float32))
    i = np.zeros((500, 1), np.int32)
    i[499] = bad
    index = CudaArray.fromNumpy(i).broadcastTo([500, 64])
    with pytest.raises(InvalidArgumentException):
        table.gather(index, 0)
    with pytest.raises(InvalidArgumentException):
        table.scatterAdd(index, CudaArray.zeros([500, 64]), 0)
