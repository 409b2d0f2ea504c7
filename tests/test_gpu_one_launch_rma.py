"""Host-initiated RMA that one launch serves: strided copies between places of the heap at every element size, and
put_signal around the sizes and alignments where the one-block form begins and ends.  Whole numbers, compared exactly
with numpy indexing; everything around the elements keeps its bytes."""
import ctypes as C

import numpy as np
import pytest

import nvshmem_amd as N
import oracle_lib as O
from gpu_util import note, runtime
from nvshmem_amd import hip

pytestmark = pytest.mark.gpu
NPES = 4
vp, sz, pd, i32, u64 = C.c_void_p, C.c_size_t, C.c_ssize_t, C.c_int, C.c_uint64


def _fn(lib, name, argtypes):
    f = getattr(lib, name)
    f.restype, f.argtypes = None, argtypes
    return f


# (elements, destination stride, source stride, bytes that both sides are off an element's alignment)
STRIDED = [(1, 1, 1, 0), (64, 1, 1, 0), (65, 3, 1, 0), (1000, 2, 5, 0), (257, 1, 7, 1), (65537, 1, 2, 0),
           (65536, 2, 1, 0), (131072, 3, 3, 0)]


@pytest.mark.parametrize("es", [1, 2, 4, 8, 16])
def test_strided_copies_in_the_heap(es):
    with runtime(NPES, 32 << 20) as rt:
        lib = rt.lib
        size = 131072 * 3 * es + 64
        a, b = rt.malloc(size), rt.malloc(size)
        A = O.fill_all("bytes", NPES, size, 7 + es)
        rt.upload_all(a, A)
        s = hip.Stream()
        iput = _fn(lib, "nvshmemx_iput%d_on_stream" % (8 * es), [vp, vp, pd, pd, sz, i32, vp])
        iget = _fn(lib, "nvshmemx_iget%d_on_stream" % (8 * es), [vp, vp, pd, pd, sz, i32, vp])
        for get in (False, True):
            for n, ds, ss, off in STRIDED:
                off = off if es > 1 else 0
                note("%s%d n=%d strides %d %d offset %d" % ("iget" if get else "iput", 8 * es, n, ds, ss, off))
                rt.fill(b, 0xEE, size)
                (iget if get else iput)(b + off, a + off, ds, ss, n, 2, s.ptr)
                s.synchronize()
                src, at = (A[2], 0) if get else (A[0], 2)
                want = np.full(size, 0xEE, np.uint8)
                k = np.arange(n)[:, None]
                lane = np.arange(es)[None, :]
                want[off + k * ds * es + lane] = src[off + k * ss * es + lane]
                assert np.array_equal(rt.download(b, at, (size,), np.uint8), want)


def test_sparse_strided_copies_and_columns():
    """Elements on lines of their own: a column of a tile to a neighbour, and more of them than the kernel takes."""
    with runtime(NPES, 64 << 20) as rt:
        lib = rt.lib
        n, stride = (1 << 17) + 1, 33
        size = n * stride * 4
        a, b = rt.malloc(size), rt.malloc(size)
        A = O.fill_all("i32", NPES, size // 4, 3)
        rt.upload_all(a, A)
        iput = _fn(lib, "nvshmem_int32_iput", [vp, vp, pd, pd, sz, i32])
        for count in (2048, n - 1, n):
            rt.fill(b, 0, size)
            iput(b, a + 4, stride, stride, count, 1)
            want = np.zeros(size // 4, np.int32)
            want[:count * stride:stride] = A[0, 1::stride][:count]
            assert np.array_equal(rt.download(b, 1, (size // 4,), np.int32), want)


@pytest.mark.parametrize("size", [1, 15, 16, 17, 1023, 1024, 8200, 65535, 65536, 65537])
def test_put_signal_in_one_launch(size):
    with runtime(NPES, 8 << 20) as rt:
        lib = rt.lib
        room = size + 64
        a, b, sig = rt.malloc(room), rt.malloc(room), rt.calloc(2, 8)
        A = O.fill_all("bytes", NPES, room, size)
        rt.upload_all(a, A)
        s = hip.Stream()
        put = _fn(lib, "nvshmemx_putmem_signal_on_stream", [vp, vp, sz, vp, u64, i32, i32, vp])
        for step, (to, frm) in enumerate([(0, 0), (1, 0), (0, 3), (5, 5), (16, 8)]):
            rt.fill(b, 0xEE, room)
            # from another PE's copy, whose address the program got from nvshmem_ptr
            put(b + to, lib.nvshmem_ptr(a, 3) + frm, size, sig, 5, N.SIGNAL_ADD, 2, s.ptr)
            put(b + to, a + frm, size, sig + 8, step, N.SIGNAL_SET, 1, s.ptr)
            s.synchronize()
            for pe, source in ((2, A[3]), (1, A[0])):
                want = np.full(room, 0xEE, np.uint8)
                want[to:to + size] = source[frm:frm + size]
                assert np.array_equal(rt.download(b, pe, (room,), np.uint8), want)
            assert rt.download(sig, 2, (2,), np.uint64).tolist() == [5 * (step + 1), 0]
            assert rt.download(sig, 1, (2,), np.uint64).tolist() == [0, step]


def test_put_signal_of_host_memory_and_refused_arguments():
    with runtime(NPES, 8 << 20) as rt:
        lib = rt.lib
        b, sig = rt.malloc(256), rt.calloc(1, 8)
        rt.fill(b, 0, 256)
        host = np.arange(100, dtype=np.uint8)
        put = _fn(lib, "nvshmemx_putmem_signal_on_stream", [vp, vp, sz, vp, u64, i32, i32, vp])
        put(b, host.ctypes.data, 100, sig, 1, N.SIGNAL_ADD, 1, None)
        rt.sync()
        assert np.array_equal(rt.download(b, 1, (100,), np.uint8), host)
        assert rt.download(sig, 1, (1,), np.uint64)[0] == 1
        put(b, b, 0, sig, 1, N.SIGNAL_ADD, 1, None)  # nothing to copy: the signal alone
        rt.sync()
        assert rt.download(sig, 1, (1,), np.uint64)[0] == 2
        put(b, b + 128, 64, sig, 1, N.SIGNAL_ADD, NPES, None)
        assert b"outside" in lib.nvshmemx_amd_last_error()
        put(b, b + 128, 64, sig, 1, 77, 2, None)
        assert b"sig_op" in lib.nvshmemx_amd_last_error()
