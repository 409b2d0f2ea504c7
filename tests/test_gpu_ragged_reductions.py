"""Reductions of buffers that start on any element: head, whole vectors and tail around 16-byte boundaries of the
destination, with the source on the same offset and on another one, in every kernel a reduction can take.  Bit for
bit against the oracle (the fold order is fixed), bytes around the destination untouched."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_util import bits_equal, note, runtime

pytestmark = pytest.mark.gpu

FORMS = {
    "gather": {"NVSHMEM_AMD_LDS_REDUCE_BYTES": str(1 << 40), "NVSHMEM_AMD_ELEMENT_REDUCE_BYTES": "0"},
    "element": {"NVSHMEM_AMD_LDS_REDUCE_BYTES": str(1 << 40), "NVSHMEM_AMD_ELEMENT_REDUCE_BYTES": str(1 << 40)},
    "lds": {"NVSHMEM_AMD_LDS_REDUCE_BYTES": "0", "NVSHMEM_AMD_TWO_STEP_REDUCE_MEMBERS": "0"},
    "two-step": {"NVSHMEM_AMD_LDS_REDUCE_BYTES": "0", "NVSHMEM_AMD_PACED_COPY_BLOCKS": "0",
                 "NVSHMEM_AMD_TWO_STEP_REDUCE_MEMBERS": "2", "NVSHMEM_AMD_TWO_STEP_REDUCE_BYTES": "0"},
}
# API type, operator, element kind, storage, (dest, source) offsets in elements
KINDS = [("int8", "min", "i8", np.int8, ((1, 1), (15, 0), (7, 12))),
         ("bfloat16", "sum", "bf16", np.uint16, ((3, 3), (7, 0), (5, 2))),
         ("float", "sum", "f32", np.float32, ((1, 1), (3, 0), (2, 3))),
         ("double", "sum", "f64", np.float64, ((1, 1), (1, 0), (0, 1)))]


def _values(kind, rng, shape):
    if kind == "i8":
        return rng.integers(-128, 128, shape, dtype=np.int8)
    x = rng.standard_normal(shape) * 10.0 ** rng.integers(-3, 4, shape)
    if kind == "bf16":
        return (x.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    return x.astype(np.float32 if kind == "f32" else np.float64)


def _guarded(got, storage, first, n):
    """The n elements from `first` on, and whether every byte around them still is 0xCD."""
    es = np.dtype(storage).itemsize
    body = np.ascontiguousarray(got[:, first * es:(first + n) * es]).view(storage)
    return body, (got[:, :first * es] == 0xCD).all() and (got[:, (first + n) * es:] == 0xCD).all()


@pytest.mark.parametrize("npes,form", [(2, "gather"), (5, "gather"), (8, "gather"), (3, "element"), (8, "element"), (16, "element"), (8, "lds"), (5, "lds"), (16, "lds"), (16, "two-step")])
def test_ragged_allreduce(npes, form, monkeypatch):
    for k, v in FORMS[form].items():
        monkeypatch.setenv(k, v)
    rng = np.random.default_rng(npes)
    with runtime(npes, 4 << 20) as rt:
        src = rt.malloc(1 << 17); dst = rt.malloc(1 << 17)
        for name, op, kind, storage, shifts in KINDS:
            vec = 16 // np.dtype(storage).itemsize
            # less than a head; a head and a tail without a vector between; around one vector and one piece; many pieces
            for n in (1, vec - 1, vec, 2 * vec - 1, 64 * vec - 1, 64 * vec + 1, 5 * 64 * vec + vec + 1):
                data = _values(kind, rng, (npes, n))
                want = O.reduce(kind, op, data)
                for d, s in shifts:
                    es = data.itemsize
                    rt.upload_all(src, data, s * es)
                    rt.fill(dst, 0xCD, n * es + 64)
                    note("%s %s %s reduce npes=%d n=%d dst+%d src+%d" % (form, name, op, npes, n, d, s))
                    rt.reduce(name, op, dst + d * es, src + s * es, n)
                    got, clean = _guarded(rt.download_all(dst, (n * es + 64,), np.uint8), storage, d, n)
                    assert clean and all(bits_equal(row, want) for row in got), (name, n, d, s)
                rt.reduce(name, op, src + s * es, src + s * es, n)   # in place, on the last source offset
                assert bits_equal(rt.download(src, npes - 1, (n,), storage, s * es), want), (name, n, s)
        rt.free(src); rt.free(dst)


@pytest.mark.parametrize("npes,form", [(2, "gather"), (8, "gather"), (16, "gather"), (3, "element"), (8, "element"), (16, "element")])
def test_ragged_reducescatter(npes, form, monkeypatch):
    for k, v in FORMS[form].items():
        monkeypatch.setenv(k, v)
    rng = np.random.default_rng(100 + npes)
    with runtime(npes, 4 << 20) as rt:
        src = rt.malloc(1 << 20); dst = rt.malloc(1 << 17)
        for name, op, kind, storage, shifts in KINDS:
            vec = 16 // np.dtype(storage).itemsize
            for n in (1, vec - 1, 2 * vec - 1, 64 * vec + 1, 3 * 64 * vec - 1):   # (every block on another offset)
                data = _values(kind, rng, (npes, npes * n))
                want = O.reducescatter(kind, op, data)
                for d, s in ((0, 0),) + shifts:
                    es = data.itemsize
                    rt.upload_all(src, data, s * es)
                    rt.fill(dst, 0xCD, n * es + 64)
                    note("%s %s reducescatter npes=%d n=%d dst+%d src+%d" % (name, op, npes, n, d, s))
                    rt.reducescatter(name, op, dst + d * es, src + s * es, n)
                    got, clean = _guarded(rt.download_all(dst, (n * es + 64,), np.uint8), storage, d, n)
                    assert clean and bits_equal(got, want), (name, n, d, s)
        rt.free(src); rt.free(dst)


@pytest.mark.parametrize("npes", [3, 8, 16])
def test_ragged_reducescatter_with_streamed_loads(npes, monkeypatch):
    """The kernels of sources that the cache cannot hold, around the ends of a piece that is cut on the source's boundaries:
    destinations on, before and behind theirs."""
    monkeypatch.setenv("NVSHMEM_AMD_CACHEABLE_SOURCE_BYTES", "0")
    monkeypatch.setenv("NVSHMEM_AMD_ELEMENT_REDUCE_BYTES", "0")
    rng = np.random.default_rng(200 + npes)
    with runtime(npes, 4 << 20) as rt:
        src = rt.malloc(1 << 20); dst = rt.malloc(1 << 17)
        for name, op, kind, storage, _ in KINDS:
            es = np.dtype(storage).itemsize
            vec = 16 // es
            for n in (vec, 63 * vec + 1, 64 * vec, 65 * vec - 1, 128 * vec + 2):
                data = _values(kind, rng, (npes, npes * n))
                want = O.reducescatter(kind, op, data)
                for d, s in ((0, 0), (0, vec - 1), (1, 0), (vec - 1, 1)):
                    rt.upload_all(src, data, s * es)
                    rt.fill(dst, 0xCD, n * es + 64)
                    note("%s %s streamed reducescatter npes=%d n=%d dst+%d src+%d" % (name, op, npes, n, d, s))
                    rt.reducescatter(name, op, dst + d * es, src + s * es, n)
                    got, clean = _guarded(rt.download_all(dst, (n * es + 64,), np.uint8), storage, d, n)
                    assert clean and bits_equal(got, want), (name, n, d, s)
        rt.free(src); rt.free(dst)


@pytest.mark.parametrize("npes,form", [(2, "gather"), (4, "lds"), (8, "lds"), (12, "lds"), (16, "lds"), (16, "two-step"), (33, "two-step")])
def test_ragged_allreduce_with_streamed_loads(npes, form, monkeypatch):
    """The kernels of sources that the cache cannot hold: source and destination on one offset in a line, on other ones a
    whole number of vectors apart and not, around the ends of a tile."""
    monkeypatch.setenv("NVSHMEM_AMD_CACHEABLE_SOURCE_BYTES", "0")
    for k, v in FORMS[form].items():
        monkeypatch.setenv(k, v)
    rng = np.random.default_rng(300 + npes)
    with runtime(npes, 2 << 20) as rt:
        src = rt.malloc(1 << 16); dst = rt.malloc(1 << 16)
        for name, op, kind, storage, _ in KINDS:
            es = np.dtype(storage).itemsize
            vec = 16 // es
            for n in (vec, 57 * vec, 64 * vec, 64 * vec + 1, 3 * 64 * vec - 1):
                data = _values(kind, rng, (npes, n))
                want = O.reduce(kind, op, data)
                for d, s in ((0, 0), (1, 1), (0, vec), (5 * vec, vec), (0, vec - 1), (vec - 1, 2)):
                    rt.upload_all(src, data, s * es)
                    rt.fill(dst, 0xCD, (n + 5 * vec) * es + 64)
                    note("%s %s %s streamed reduce npes=%d n=%d dst+%d src+%d" % (form, name, op, npes, n, d, s))
                    rt.reduce(name, op, dst + d * es, src + s * es, n)
                    got, clean = _guarded(rt.download_all(dst, ((n + 5 * vec) * es + 64,), np.uint8), storage, d, n)
                    assert clean and all(bits_equal(row, want) for row in got), (name, n, d, s)
                rt.reduce(name, op, src + s * es, src + s * es, n)   # in place
                assert bits_equal(rt.download(src, npes - 1, (n,), storage, s * es), want), (name, n, s)
        rt.free(src); rt.free(dst)


@pytest.mark.parametrize("cacheable", ["none", "all"])
@pytest.mark.parametrize("npes,form", [(2, "gather"), (3, "gather"), (4, "lds"), (8, "lds"), (12, "lds"), (16, "lds")])
def test_ragged_allreduce_whose_tiles_share_lines(npes, form, cacheable, monkeypatch):
    """Streamed sources on another offset in a line than the destination, in the sizes where the lanes at a tile's ends load
    cacheable (the cache could hold them: 2/3 of it) and beyond: fewer tiles than are dealt to the XCDs, and a round of 32 of
    them with some left over."""
    for k, v in FORMS[form].items():
        monkeypatch.setenv(k, v)
    for nbytes in (1024 + 8, 41 * 1024 + 8):   # of every PE, whatever the element type
        monkeypatch.setenv("NVSHMEM_AMD_CACHEABLE_SOURCE_BYTES", "0" if cacheable == "none" else str(npes * nbytes * 3 // 2))
        rng = np.random.default_rng(npes * nbytes)
        with runtime(npes, 2 << 20) as rt:
            src = rt.malloc(1 << 16); dst = rt.malloc(1 << 16)
            for name, op, kind, storage, _ in KINDS:
                es = np.dtype(storage).itemsize
                vec, n = 16 // es, nbytes // es
                data = _values(kind, rng, (npes, n))
                want = O.reduce(kind, op, data)
                for d, s in ((0, 0), (0, vec), (5 * vec, vec), (0, vec - 1), (vec - 1, 2)):
                    rt.upload_all(src, data, s * es)
                    rt.fill(dst, 0xCD, (n + 5 * vec) * es + 64)
                    note("%s %s %s shared lines npes=%d n=%d dst+%d src+%d %s" % (form, name, op, npes, n, d, s, cacheable))
                    rt.reduce(name, op, dst + d * es, src + s * es, n)
                    got, clean = _guarded(rt.download_all(dst, ((n + 5 * vec) * es + 64,), np.uint8), storage, d, n)
                    assert clean and all(bits_equal(row, want) for row in got), (name, n, d, s)
            rt.free(src); rt.free(dst)
