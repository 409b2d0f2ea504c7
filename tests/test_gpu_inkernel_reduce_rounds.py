"""GPU parity of the in-kernel allreduce's fold of whole vectors, at the sizes where its rounds change: fewer vectors than
lanes, remainders of every kind of round, 16 vectors per lane, the first size of rounds that the block's wavefronts go
through together, and team sizes on either side of the numbers of members fetched at a time."""
import numpy as np
import pytest

import nvshmem_amd as N
import oracle_lib as O
from gpu_util import bits_equal, note, runtime

pytestmark = pytest.mark.gpu

PHASED_BYTES, MANY = 512 << 10, 16


def _data(kind, shape, rng):
    if kind == "bf16":
        return (rng.standard_normal(shape).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    return rng.standard_normal(shape).astype(O.NP_STORAGE[kind])


def _slices(npes, threads):
    """Whole vectors that one PE folds."""
    phased = -(-PHASED_BYTES // (16 * npes))
    return sorted({1, threads - 1, threads + 1, 3 * threads + 5, MANY * threads - 1, MANY * threads + threads // 2 + 3,
                   phased - 1, phased, phased + 2 * threads + 7})


@pytest.mark.parametrize("npes", [2, 3, 5, 8, 9, 16, 17])
@pytest.mark.parametrize("threads", [64, 320, 512, 1024])
def test_rounds_at_their_edges(npes, threads):
    rng = np.random.default_rng(npes * 2048 + threads)
    slices = _slices(npes, threads)
    room = (max(slices) * npes + 1) * 16
    with runtime(npes, 2 * room + (8 << 20)) as rt:
        perf = rt.perftest()
        src, dst = rt.malloc(room), rt.malloc(room)
        for i, nvec in enumerate(slices):
            kind, op = [("f32", "sum"), ("bf16", "sum"), ("f32", "max")][i % 3]
            per = 16 // np.dtype(O.NP_STORAGE[kind]).itemsize
            n = nvec * npes * per - (i % 2)  # every second one ends inside a vector
            data = _data(kind, (npes, n), rng)
            rt.upload_all(src, data)
            want = O.reduce(kind, op, data)
            for to in (dst, src):  # in place too
                note("device reduce %s %s npes=%d threads=%d n=%d" % (kind, op, npes, threads, n))
                assert perf.nvshmem_perftest_device_reduce(N.DTYPES[kind], N.OPS[op], to, src, n, N.SCOPE_BLOCK, threads, None) == 0
                rt.sync()
                got = rt.download_all(to, (n,), data.dtype)
                for pe in range(npes):
                    assert bits_equal(got[pe], want), (kind, op, n, pe)


@pytest.mark.parametrize("npes", [4, 8, 16, 24])
@pytest.mark.parametrize("threads", [64, 100, 256, 1024])
def test_rounds_that_fetch_the_next_ahead_of_their_stores(npes, threads):
    """Teams of a whole number of members a round fetches: no round, one, two and three of them, short of a round by one
    vector and one vector beyond; in place, where the next round is fetched before this one is written."""
    rng = np.random.default_rng(npes * 4096 + threads)
    per_round = threads * (2 if npes == 4 else 1)
    room = (3 * per_round + 2) * npes * 16
    with runtime(npes, 2 * room + (8 << 20)) as rt:
        perf = rt.perftest()
        src, dst = rt.malloc(room), rt.malloc(room)
        for rounds in (1, 2, 3):
            for nvec in (rounds * per_round - 1, rounds * per_round, rounds * per_round + 1):
                for kind, op in (("f32", "sum"), ("bf16", "max"), ("bf16", "sum")):
                    n = nvec * npes * (16 // np.dtype(O.NP_STORAGE[kind]).itemsize)
                    data = _data(kind, (npes, n), rng)
                    want = O.reduce(kind, op, data)
                    rt.upload_all(src, data)
                    for to in (dst, src):
                        note("device reduce %s %s npes=%d threads=%d n=%d" % (kind, op, npes, threads, n))
                        assert perf.nvshmem_perftest_device_reduce(N.DTYPES[kind], N.OPS[op], to, src, n, N.SCOPE_BLOCK, threads, None) == 0
                        rt.sync()
                        got = rt.download_all(to, (n,), data.dtype)
                        assert all(bits_equal(row, want) for row in got), (kind, op, n)
