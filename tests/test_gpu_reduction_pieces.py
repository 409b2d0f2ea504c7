"""Reductions of more than a single launch can hold."""
import numpy as np
import pytest

from gpu_util import note, runtime

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npes,doff,soff", [(4, 3, 3), (2, 1, 2)])
def test_ragged_allreduce_of_more_than_one_launch(npes, doff, soff):
    """Reductions go out in pieces of 2 GiB per PE; nothing is missing or added twice where two of them meet, wherever the
    buffers start."""
    n = (1 << 29) + (1 << 20) + 5                      # int32: one whole piece and a short one
    windows = (0, (1 << 29) - 2048, n - 4096)           # where the data differs from element to element
    rng = np.random.default_rng(npes)
    with runtime(npes, 2 * (4 * n + 64) + (64 << 20)) as rt:
        src = rt.malloc(4 * n + 64); dst = rt.malloc(4 * n + 64)
        rt.fill(src, 0x01, 4 * n + 64); rt.fill(dst, 0xCD, 4 * n + 64)
        rt.sync()
        want = np.full(n, 0x01010101 * npes, np.int32)
        for at in windows:
            part = rng.integers(-2**28, 2**28, (npes, 4096), dtype=np.int32)
            rt.upload_all(src, part, (soff + at) * 4)
            want[at:at + 4096] = part.sum(axis=0)
        note("int32 sum reduce of %d elements on %d PEs, dst+%d src+%d" % (n, npes, doff, soff))
        rt.reduce("int32", "sum", dst + 4 * doff, src + 4 * soff, n)
        for pe in (0, npes - 1):
            got = rt.download(dst, pe, (4 * n + 64,), np.uint8)
            assert np.array_equal(got[4 * doff:4 * (doff + n)].view(np.int32), want)
            assert (got[:4 * doff] == 0xCD).all() and (got[4 * (doff + n):] == 0xCD).all()
