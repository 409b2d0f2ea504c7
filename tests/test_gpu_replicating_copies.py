"""fcollect and broadcast store every piece to all members, back to back or one destination after the other: both ways
at every remainder of the unrolled stores and around the edges of vectors and pieces, byte for byte against the oracle
with the bytes around the destination untouched; and alltoall over the same sizes."""
import numpy as np
import pytest

import nvshmem_amd as N
import oracle_lib as O
from gpu_util import note, runtime

pytestmark = pytest.mark.gpu

SIZES = (1, 15, 31, 1023, 1024, 1041, 3 * 1024 + 17, 70001)
OFFSETS = ((0, 0), (3, 3), (5, 16), (16, 9))     # (destination, source) within the allocations


@pytest.mark.parametrize("blocks", ["0", str(1 << 40)])      # NVSHMEM_AMD_PACED_COPY_BLOCKS: one by one, back to back
@pytest.mark.parametrize("npes", [2, 3, 5, 8, 12, 15, 64])
def test_copies_to_every_member(npes, blocks, monkeypatch):
    monkeypatch.setenv("NVSHMEM_AMD_PACED_COPY_BLOCKS", blocks)
    rng = np.random.default_rng(npes)
    with runtime(npes, 14 << 20) as rt:
        top = max(SIZES)
        src = rt.malloc(npes * top + 64); dst = rt.malloc(npes * top + 64)
        for n in SIZES:
            data = rng.integers(0, 256, (npes, npes * n), dtype=np.uint8)
            one = np.ascontiguousarray(data[:, :n])
            for doff, soff in OFFSETS:
                rt.upload_all(src, data, soff)
                note("npes=%d n=%d dst+%d src+%d paced from %s blocks" % (npes, n, doff, soff, blocks))
                for what, nbytes, want in (("fcollect", npes * n, O.fcollect(one)), ("broadcast", n, O.broadcast(one, npes - 1)),
                                           ("alltoall", npes * n, O.alltoall(data))):
                    rt.fill(dst, 0xCD, nbytes + 64)
                    if what == "broadcast":
                        rt.broadcastmem(dst + doff, src + soff, n, npes - 1)
                    else:
                        (rt.fcollectmem if what == "fcollect" else rt.alltoallmem)(dst + doff, src + soff, n)
                    got = rt.download_all(dst, (nbytes + 64,), np.uint8)
                    assert np.array_equal(got[:, doff:doff + nbytes], want), (what, n, doff, soff)
                    assert (got[:, :doff] == 0xCD).all() and (got[:, doff + nbytes:] == 0xCD).all(), (what, n, doff, soff)
        rt.free(src); rt.free(dst)


def test_alltoall_of_a_family_of_teams():
    """One launch for all rows, or all columns, of a 2-D split with a short last row: the team is read from the table."""
    npes, xr, n = 14, 4, 1041
    rng = np.random.default_rng(5)
    with runtime(npes, 4 << 20) as rt:
        src = rt.malloc(npes * n); dst = rt.malloc(npes * n)
        xt, yt = rt.team_split_2d(N.TEAM_WORLD, xr)
        families = ((xt, [list(range(r, min(r + xr, npes))) for r in range(0, npes, xr)]),
                    (yt, [list(range(c, npes, xr)) for c in range(xr)]))
        for team, rows in families:
            data = rng.integers(0, 256, (npes, npes * n), dtype=np.uint8)
            rt.upload_all(src, data)
            note("alltoall of %d teams" % len(rows))
            rt.alltoallmem(dst, src, n, team=team)
            for members in rows:
                want = O.alltoall(np.ascontiguousarray(data[members][:, :len(members) * n]))
                for k, pe in enumerate(members):
                    assert np.array_equal(rt.download(dst, pe, (len(members) * n,), np.uint8), want[k]), (members, pe)
        rt.team_destroy(xt); rt.team_destroy(yt)
        rt.free(src); rt.free(dst)


@pytest.mark.parametrize("npes", [2, 8, 16])
def test_segments_around_the_order_of_edges_and_vectors(npes):
    """Short segments store their edge bytes before the vectors, longer ones behind them; segments of one PE touch those
    of its neighbours in the middle of a vector."""
    rng = np.random.default_rng(50 + npes)
    with runtime(npes, 2 << 20) as rt:
        src = rt.malloc(npes * 1100 + 64); dst = rt.malloc(npes * 1100 + 64)
        for n in (16, 17, 33, 511, 512, 513, 1039):
            data = rng.integers(0, 256, (npes, npes * n), dtype=np.uint8)
            one = np.ascontiguousarray(data[:, :n])
            for doff, soff in OFFSETS:
                rt.upload_all(src, data, soff)
                note("npes=%d n=%d dst+%d src+%d" % (npes, n, doff, soff))
                for what, nbytes, want in (("fcollect", npes * n, O.fcollect(one)), ("broadcast", n, O.broadcast(one, 1)),
                                           ("alltoall", npes * n, O.alltoall(data))):
                    rt.fill(dst, 0xCD, nbytes + 64)
                    if what == "broadcast":
                        rt.broadcastmem(dst + doff, src + soff, n, 1)
                    else:
                        (rt.fcollectmem if what == "fcollect" else rt.alltoallmem)(dst + doff, src + soff, n)
                    got = rt.download_all(dst, (nbytes + 64,), np.uint8)
                    assert np.array_equal(got[:, doff:doff + nbytes], want), (what, n, doff, soff)
                    assert (got[:, :doff] == 0xCD).all() and (got[:, doff + nbytes:] == 0xCD).all(), (what, n, doff, soff)
        rt.free(src); rt.free(dst)
