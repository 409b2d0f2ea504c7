"""Collective launches on several streams run one after the other, whichever way each is started: small grids with a
plain launch, grids of more than half of the GPU cooperatively.  Every kernel here waits for the other PEs inside
itself, on state of its own, so two of them holding part of the GPU each would give up and be counted."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_util import note, runtime
from nvshmem_amd import hip

pytestmark = pytest.mark.gpu

NPES, CHUNK, ROUNDS = 8, 64, 20


@pytest.mark.parametrize("forced", [None, "0", "1"])     # by size; always cooperative; always plain (one stream only)
def test_collective_launches_on_two_streams(forced, monkeypatch):
    if forced is None:
        monkeypatch.delenv("NVSHMEM_AMD_PLAIN_COLLECTIVE_LAUNCH", raising=False)
    else:
        monkeypatch.setenv("NVSHMEM_AMD_PLAIN_COLLECTIVE_LAUNCH", forced)
    with runtime(NPES, 32 << 20) as rt:
        perf = rt.perftest()
        first = hip.Stream()
        streams = (first, first if forced == "1" else hip.Stream(), hip.Stream() if forced is None else first)
        jobs = []
        for k, blocks in enumerate((4, 200, 64)):        # 200 blocks of 256 threads per PE: most of the GPU
            n = blocks * CHUNK * 2
            data = O.fill_all("i32", NPES, n, 40 + k)
            src, dst, sig = rt.malloc(n * 4), rt.calloc(n, 4), rt.calloc(blocks, 8)
            counter, errors = rt.calloc(1, 8), rt.calloc(1, 8)
            rt.upload_all(src, data)
            jobs.append((blocks, n, src, dst, sig, counter, errors, data))
        rt.sync()
        before = rt.lib.nvshmemx_amd_timeout_count()
        note("collective launches of 4, 200 and 64 blocks per PE on several streams, forced=%s" % forced)
        for i in range(3 * ROUNDS):
            blocks, n, src, dst, sig, counter, errors, _ = jobs[i % 3]
            # (all barriers meet on the one row of the world team: overlapping launches would also disturb them)
            s = streams[i % 3].ptr
            assert perf.nvshmem_perftest_ring_reduce(dst, src, n, sig, CHUNK, blocks, 256, s) == 0
            assert perf.nvshmem_perftest_device_barrier(counter, errors, 5, 2, 256, s) == 0
        rt.sync()
        assert rt.lib.nvshmemx_amd_timeout_count() == before
        for blocks, n, src, dst, sig, counter, errors, data in jobs:
            assert (rt.download_all(dst, (n,), np.int32) == O.reduce("i32", "sum", data)).all()
            assert (rt.download_all(errors, (1,), np.uint64) == 0).all()
        for s in set(streams):
            s.destroy()


def test_captured_launch_behind_plain_ones():
    """A collective launch is captured while plain ones on another stream are still on their way; every replay and the
    launches between the replays give what they give on a stream."""
    with runtime(NPES, 32 << 20) as rt:
        perf = rt.perftest()
        s, other = hip.Stream(), hip.Stream()
        n, blocks = 8 * CHUNK * 2, 8
        src, dst, sig = rt.malloc(n * 4), rt.calloc(n, 4), rt.calloc(blocks, 8)
        eager, eager_sig = rt.calloc(n, 4), rt.calloc(blocks, 8)
        rt.upload_all(src, O.fill_all("i32", NPES, n, 7))
        rt.sync()
        before = rt.lib.nvshmemx_amd_timeout_count()
        for _ in range(ROUNDS):
            assert perf.nvshmem_perftest_ring_reduce(eager, src, n, eager_sig, CHUNK, blocks, 256, other.ptr) == 0
        with hip.Graph(s) as g:
            assert perf.nvshmem_perftest_ring_reduce(dst, src, n, sig, CHUNK, blocks, 256, s.ptr) == 0
        for k in range(3):
            data = O.fill_all("i32", NPES, n, 50 + k)
            note("replay %d" % k)
            rt.upload_all(src, data)
            rt.sync()
            g.launch()
            assert perf.nvshmem_perftest_ring_reduce(eager, src, n, eager_sig, CHUNK, blocks, 256, s.ptr) == 0
            s.synchronize()
            want = O.reduce("i32", "sum", data)
            assert (rt.download_all(dst, (n,), np.int32) == want).all()
            assert (rt.download_all(eager, (n,), np.int32) == want).all()
        assert rt.lib.nvshmemx_amd_timeout_count() == before
        g.destroy()
        for x in (s, other):
            x.destroy()
