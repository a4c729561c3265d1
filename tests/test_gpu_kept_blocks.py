"""Freed blocks kept for the runtime stream's next allocations: a block comes
back for the same rounded size, never while it is held, never into or out of a
stream capture, and stays within the bound; threads that share the stream keep
their values."""
import ctypes
import threading

import numpy as np
import pytest

from phptensors import _abi as A

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    L = A.load()
    A.check(L.pt_init(), "init")
    yield L
    A.check(L.pt_mem_init(0), "bound")


def _alloc(lib, nbytes, stream=None):
    p = ctypes.c_void_p()
    A.check(lib.pt_alloc(ctypes.byref(p), nbytes, stream), "alloc")
    return p.value


def _kept(lib):
    size, count = ctypes.c_size_t(), ctypes.c_size_t()
    A.check(lib.pt_mem_kept(ctypes.byref(size), ctypes.byref(count)))
    return size.value, count.value


@pytest.mark.parametrize("nbytes", [1, 511, 512, 513, 8191, 8192, 8193, 100000, 1 << 20, (1 << 20) + 1, 50_000_001])
def test_block_returns_for_its_size_only(lib, nbytes):
    p = _alloc(lib, nbytes)
    A.check(lib.pt_free(p, None))
    q = _alloc(lib, nbytes)
    assert q == p
    r = _alloc(lib, nbytes)  # p is held: another block
    assert r != q and abs(r - q) >= nbytes
    x = np.arange(nbytes % 251 + 1, dtype=np.uint8)[:nbytes]
    A.check(lib.pt_memcpy_h2d(q, x.ctypes.data, x.nbytes, None))
    A.check(lib.pt_memset(r, 7, nbytes, None))
    y = np.empty_like(x)
    A.check(lib.pt_memcpy_d2h(y.ctypes.data, q, y.nbytes, None))
    assert np.array_equal(x, y)
    # bigger than twice the block: never served from it
    A.check(lib.pt_free(q, None))
    s = _alloc(lib, 4 * nbytes + 4096)
    assert s != q
    for b in (r, s):
        A.check(lib.pt_free(b, None))


def test_other_streams_and_captures_pass_by(lib):
    """A block freed on another stream is not kept; a capture of the runtime
    stream neither takes nor gives blocks, and its replays stay right while
    eager work reuses everything that is kept."""
    stream = ctypes.c_void_p()
    A.check(lib.pt_stream_create(ctypes.byref(stream)))
    p = _alloc(lib, 70000)
    A.check(lib.pt_stream_synchronize(None))
    before = _kept(lib)
    A.check(lib.pt_free(p, stream))
    assert _kept(lib) == before
    p = _alloc(lib, 70000, stream)
    A.check(lib.pt_stream_synchronize(stream))
    A.check(lib.pt_free(p, None))  # allocated on the other stream
    assert _kept(lib) == before
    q = _alloc(lib, 70000)
    before = _kept(lib)
    A.check(lib.pt_free(q, None))
    assert _kept(lib) == (before[0] + 73728, before[1] + 1)
    A.check(lib.pt_stream_synchronize(stream))
    A.check(lib.pt_stream_destroy(stream))

    rng = np.random.default_rng(3)
    x = np.round(rng.uniform(-8, 8, (9000, 40))).astype(np.float32)
    dx, out = A.to_device(x), A.DeviceBuffer(160)
    shape, strides = A.ints(x.shape), A.sizes([40, 1])
    op = A.OP["sum"]

    def reduce():  # splits the rows: its scratch comes from the pool, or from the graph
        A.check(lib.pt_reduce(dx.ptr, out.ptr, A.FLOAT32, op, shape, strides, 2, 0, 0, None), "sum")

    reduce()
    graph = ctypes.c_void_p()
    before = _kept(lib)
    A.check(lib.pt_graph_begin_capture(None))
    reduce()
    A.check(lib.pt_graph_end_capture(None, ctypes.byref(graph)))
    assert _kept(lib) == before
    for i in range(6):
        A.check(lib.pt_memset(out.ptr, 0xFF, 160, None))
        A.check(lib.pt_graph_launch(graph, None))
        junk = [A.DeviceBuffer(n) for n in (40 * 128 * 4, 20480, 512, 100000)]
        for j in junk:
            A.check(lib.pt_memset(j.ptr, 0xFF, j.nbytes, None))
        assert np.array_equal(out.download(np.float32, (40,)), x.sum(0)), i
        for j in junk:
            j.free()
    A.check(lib.pt_graph_destroy(graph))


def test_bound(lib):
    """Blocks in use and kept together stay within the threshold, or none are
    kept, and the threshold can be lowered."""
    A.check(lib.pt_mem_init(1))
    assert _kept(lib) == (0, 0)
    A.check(lib.pt_free(_alloc(lib, 300_000), None))
    assert _kept(lib) == (0, 0)
    A.check(lib.pt_mem_init(1 << 34))
    blocks = [_alloc(lib, 300_000) for _ in range(8)]
    assert len(set(blocks)) == 8
    for i, b in enumerate(blocks):
        A.check(lib.pt_free(b, None))
        assert _kept(lib) == ((i + 1) * 327680, i + 1)
    again = [_alloc(lib, 300_000) for _ in range(8)]
    assert set(again) == set(blocks) and _kept(lib) == (0, 0)
    for b in again[:4]:
        A.check(lib.pt_free(b, None))
    A.check(lib.pt_mem_init(3 * 327680))  # with the four in use
    assert _kept(lib) == (0, 0)
    for b in again[4:]:
        A.check(lib.pt_free(b, None))
        assert _kept(lib)[0] <= 3 * 327680
    A.check(lib.pt_mem_init(0))


def test_failed_allocation_gives_back(lib):
    """More than the card holds: refused, after every kept block went back to the driver's pool."""
    total = ctypes.c_size_t()
    A.check(lib.pt_mem_info(None, ctypes.byref(total), None))
    stream = ctypes.c_void_p()
    A.check(lib.pt_stream_create(ctypes.byref(stream)))
    for st in (None, stream):
        A.check(lib.pt_free(_alloc(lib, 1 << 20), None))
        assert _kept(lib)[1] > 0
        p = ctypes.c_void_p()
        assert lib.pt_alloc(ctypes.byref(p), 4 * total.value, st) == A.PT_ERR_NOMEM and not p.value
        assert _kept(lib) == (0, 0)
        x = A.to_device(np.arange(100, dtype=np.float32))
        assert np.array_equal(x.download(np.float32, (100,)), np.arange(100))
        x.free()
    A.check(lib.pt_stream_destroy(stream))


@pytest.mark.parametrize("nbytes", [2 ** 63, 2 ** 63 + 1, 2 ** 64 - 512, 2 ** 64 - 1])
def test_sizes_that_cannot_exist_are_refused(lib, nbytes):
    p = ctypes.c_void_p()
    assert lib.pt_alloc(ctypes.byref(p), nbytes, None) == A.PT_ERR_NOMEM and not p.value
    A.check(lib.pt_free(_alloc(lib, 1000), None))


@pytest.mark.parametrize("shape", [(2000000000, 2000000000), (65536, 65536, 65536, 16384), (65536, 65536, 65536, 16385)],
                         ids=str)
def test_tensors_that_cannot_exist_are_refused(lib, shape):
    """16 EB, and bytes that wrap to 0 and to 1 PiB in 64 bits."""
    from phptensors import CudaArray
    with pytest.raises(A.RuntimeException, match="allocation"):
        CudaArray.zeros(list(shape))
    assert CudaArray.full([3], 2.0).toNumpy().tolist() == [2.0] * 3


def test_threads_share_the_stream(lib):
    from phptensors import CudaArray
    errors = []

    def work(k):
        try:
            for i in range(200):
                n = 1000 + 37 * ((i + k) % 5)
                a = CudaArray.full([n], float(k + 1))
                b = a * 3.0 + a
                if i % 20 == 0 and not np.all(b.toNumpy() == 4.0 * (k + 1)):
                    errors.append((k, i))
                del a, b
        except Exception as exc:  # reported by the main thread
            errors.append((k, repr(exc)))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not any(t.is_alive() for t in threads) and not errors, errors[:3]
