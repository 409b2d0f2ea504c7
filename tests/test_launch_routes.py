"""Which kernels the library launches for a call, and with which grids: seen on the CPU, where nothing runs."""
import pytest

from launch_recorder import recorded  # noqa: F401

COLLECTIVE_LAUNCH = """
ok(lib.nvshmemx_amd_init(8, 1 << 20))
launches()
for threads, blocks in ((64, 1), (1024, 1), (256, 32), (256, 200)):
    for stream in (None, 1, 2, 1):
        ok(lib.nvshmemx_amd_collective_launch(1, blocks, 1, 1, threads, 1, 1, None, 0, stream))
for kernel, cooperative, grid, block, lds in launches():
    assert cooperative == %s, (grid, block)
    assert grid[2] == 8
"""


@pytest.mark.parametrize("plain,cooperative", [(None, True), ("0", True), ("1", False)])
def test_collective_launches_are_cooperative_unless_asked(recorded, plain, cooperative):  # noqa: F811
    """Only the cooperative queue keeps a PE kernel apart from cooperative kernels that the program itself has on
    another stream: side by side, each could hold compute units that the other waits for."""
    env = {} if plain is None else {"NVSHMEM_AMD_PLAIN_COLLECTIVE_LAUNCH": plain}
    recorded(COLLECTIVE_LAUNCH % cooperative, **env)


@pytest.mark.parametrize("scope", [1, 2, 1 | 256, 2 | 256 | 512])
def test_token_dispatch_sends_and_waits_in_plain_launches(recorded, scope):  # noqa: F811
    """Blocks that send never wait, so neither launch needs its grid to be resident as a whole; grids that could not be
    are refused all the same."""
    recorded("""
perf = _lib.load_perftest()
ok(lib.nvshmemx_amd_init(8, 8 << 20))
a = lib.nvshmem_malloc(1 << 20)
launches()
def dispatch(blocks):
    return perf.nvshmem_perftest_moe_dispatch_put_signal(a, 8, a, a, a, a, a, 1, 8, 2, 1024, blocks, 256, %d, None)
assert dispatch(64) == 0
(sender, c0, grid, block, lds), (receiver, c1, wait_grid, wait_block, lds1) = launches()
assert "moe_dispatch" in sender and not c0 and grid == (64, 1, 8) and block == (256, 1, 1)
assert "moe_receive" in receiver and not c1 and wait_grid == (1, 1, 8) and wait_block == (64, 1, 1)
assert dispatch(1 << 20) != 0 and not launches()
""" % scope)


@pytest.mark.parametrize("scope,full", [(1 | 256, True), (2 | 256, False)])
def test_full_size_dispatch_of_wavefronts_holds_its_stores_back(recorded, scope, full):  # noqa: F811
    """More than 1 GiB of row copies, all PEs together."""
    recorded("""
perf = _lib.load_perftest()
ok(lib.nvshmemx_amd_init(8, 32 << 20))
a = lib.nvshmem_malloc(16 << 20)
def sender(tokens):
    launches()
    assert perf.nvshmem_perftest_moe_dispatch_put_signal(a, 8, a, a, a, a, a, 1, tokens, 64, 16384, 64, 256, %d, None) == 0
    return launches()[0][0]
assert ("ILb1ELb1E" in sender(129)) == %s
assert "ILb1ELb1E" not in sender(128)
""" % (scope, full))


def test_copies_that_are_in_flight_all_at_once_are_not_paced(recorded):  # noqa: F811
    """fcollect and broadcast of up to 32 pieces per compute unit (16 from 12 members on) store back to back, larger ones
    one destination at a time (third template argument of the kernel)."""
    recorded("""
for npes in (4, 8, 16):
    ok(lib.nvshmemx_amd_init(npes, 256 << 20))
    a, b = lib.nvshmem_malloc(64 << 20), lib.nvshmem_malloc(128 << 20)
    launches()
    for blocks, paced in ((1, 0), (4096, 0), (5000, npes >= 12), (8192, npes >= 12), (8700, 1), (20000, 1)):
        ok(lib.nvshmemx_fcollectmem_on_stream(0, b, a, blocks // npes * 1024 or 1, None))
        ok(lib.nvshmemx_broadcastmem_on_stream(0, b, a, blocks * 1024 - 5, 1, None))
        for kernel, cooperative, grid, block, lds in launches():
            assert "ELb%dELi" % paced in kernel and (lds > 0) == bool(paced), (npes, blocks, kernel, lds)
    lib.nvshmem_finalize()
""")


def test_wavefronts_of_paced_copies(recorded):  # noqa: F811
    """A compute unit (160 KiB of LDS) holds 16 wavefronts of a paced copy whose sources the cache holds, more with
    streamed loads (second template argument)."""
    recorded("""
for npes, mib, streamed, waves in ((8, 32, 0, 16), (16, 16, 0, 16), (16, 8, 0, 16), (8, 64, 1, 24), (12, 32, 1, 28)):
    ok(lib.nvshmemx_amd_init(npes, (npes + 2) * mib << 20))
    a, b = lib.nvshmem_malloc(mib << 20), lib.nvshmem_malloc(npes * mib << 20)
    launches()
    ok(lib.nvshmemx_fcollectmem_on_stream(0, b, a, mib << 20, None))
    (kernel, _, grid, block, lds), = launches()
    assert "ILi0ELb%dELb1E" % streamed in kernel and (160 << 10) // lds == waves, (npes, mib, kernel, lds)
    lib.nvshmem_finalize()
""")


@pytest.mark.parametrize("npes,gib", [(8, 9), (3, 18), (16, 5), (2, 65), (1, 65)])
def test_the_largest_reductions_are_launched_whole(recorded, npes, gib):  # noqa: F811
    """No launch of 2^32 threads or more, however long and ragged the buffers are: every element in one piece or another."""
    recorded("""
npes, nbytes = %d, %d << 30
ok(lib.nvshmemx_amd_init(npes, nbytes + (1 << 30)))
a = lib.nvshmem_malloc(nbytes + 64)
launches()
for name, es in (("float", 4), ("bfloat16", 2), ("double", 8)):
    n = nbytes // es - 3
    ok(_lib.typed_coll(lib, "nvshmemx_%%s_sum_reduce_on_stream" %% name, True)(0, a + es, a + es, n, None))
    vectors = sum((grid[0] - 2) * 64 for kernel, _, grid, block, lds in launches() if "reduce_" in kernel)
    assert n * es // 16 - 4096 <= vectors <= n * es // 16 + 64, (name, vectors)
if npes == 1:
    b = lib.nvshmem_malloc(1 << 20)
    fn = _lib.typed_coll(lib, "nvshmemx_float_sum_reducescatter_on_stream", True)
    ok(lib.nvshmem_finalize() or lib.nvshmemx_amd_init(1, 2 * nbytes + (1 << 30)))
    a, b = lib.nvshmem_malloc(nbytes + 64), lib.nvshmem_malloc(nbytes + 64)
    launches()
    ok(fn(0, b + 4, a + 8, nbytes // 4 - 3, None))
    assert sum(grid[0] * 64 for _, _, grid, _, _ in launches()) >= nbytes // 16 - 4096
""" % (npes, gib))


def test_small_ragged_reductions_fold_an_element_per_lane(recorded):  # noqa: F811
    """Ragged buffers with up to 512 KiB of results, but for the types and team sizes that the vector kernels serve faster;
    aligned buffers never."""
    recorded("""
ELEMENT, VECTOR = True, False
for npes, kind, name, nbytes, shift, element in (
        (16, "reduce", "int8", 65537, 1, ELEMENT), (16, "reduce", "int8", 1 << 19, 1, ELEMENT), (16, "reduce", "int8", (1 << 19) + 1, 1, VECTOR),
        (16, "reduce", "int8", 65536, 0, VECTOR), (16, "reduce", "float", 4100, 1, VECTOR), (3, "reduce", "float", 4100, 1, ELEMENT),
        (2, "reduce", "double", 4104, 1, ELEMENT), (8, "reduce", "bfloat16", 8192, 1, ELEMENT), (8, "reduce", "bfloat16", 8194, 1, VECTOR),
        (8, "reduce", "float", 404, 1, VECTOR), (4, "reduce", "int8", 100, 1, ELEMENT), (4, "reduce", "int8", 10000, 1, VECTOR),
        (16, "reducescatter", "float", 32768, 1, ELEMENT), (16, "reducescatter", "float", 32772, 0, VECTOR),
        (16, "reducescatter", "float", 32764, 0, ELEMENT), (16, "reducescatter", "float", 32752, 0, VECTOR),
        (8, "reducescatter", "int8", 4095, 0, ELEMENT), (8, "reducescatter", "int8", 4097, 0, VECTOR), (8, "reducescatter", "float", 404, 0, VECTOR)):
    es = {"int8": 1, "bfloat16": 2, "float": 4, "double": 8}[name]
    ok(lib.nvshmemx_amd_init(npes, 32 << 20))
    a, b = lib.nvshmem_malloc(16 << 20), lib.nvshmem_malloc(1 << 20)
    launches()
    ok(_lib.typed_coll(lib, "nvshmemx_%s_max_%s_on_stream" % (name, kind), True)(0, b + shift * es, a + shift * es, nbytes // es, None))
    (kernel, _, grid, block, _), = launches()
    assert ("reduce_element_kernel" in kernel) == element, (npes, kind, name, nbytes, shift, kernel)
    assert not element or (grid[0] - 1) * block[0] < nbytes // es <= grid[0] * block[0]
    lib.nvshmem_finalize()
""")


def test_streamed_fcollects_of_many_members_walk_in_chunks(recorded):  # noqa: F811
    """From 16 members on (fifth template argument): whole chunks, every tile of a segment for each group of members."""
    recorded("""
for npes, mib, groups in ((15, 40, 0), (16, 16, 0), (16, 24, 8), (24, 16, 8), (64, 5, 32)):
    ok(lib.nvshmemx_amd_init(npes, (npes + 2) * mib << 20))
    a, b = lib.nvshmem_malloc(mib << 20), lib.nvshmem_malloc(npes * mib << 20)
    launches()
    ok(lib.nvshmemx_fcollectmem_on_stream(0, b, a, (mib << 20) - 5, None))
    (kernel, _, grid, block, lds), = launches()
    assert ("ELi2ELb1EE" in kernel) == bool(groups), (npes, mib, kernel)
    assert not groups or (grid[0] % 16384 == 0 and grid[0] // groups >= mib * 1024 > grid[0] // groups - 16384 // groups - 2)
    lib.nvshmem_finalize()
""")


def test_large_sources_of_reductions_are_streamed(recorded):  # noqa: F811
    """More than 96 MiB of sources, all PEs together, take the kernels with streamed loads; an eighth of them being 1- or
    2-byte elements then has a wavefront of its own."""
    recorded("""
ok(lib.nvshmemx_amd_init(8, 64 << 20))
a, b = lib.nvshmem_malloc(16 << 20), lib.nvshmem_malloc(16 << 20)
for name, es in (("float", 4), ("bfloat16", 2)):
    for over in (0, 1):
        n = (12 << 20) // es + over
        launches()
        ok(_lib.typed_coll(lib, "nvshmemx_%s_sum_reduce_on_stream" % name, True)(0, b, a, n, None))
        ok(_lib.typed_coll(lib, "nvshmemx_%s_sum_reducescatter_on_stream" % name, True)(0, b, a, (12 << 20) // 8 // es + over, None))
        (reduce, _, _, block, _), (scatter, _, _, _, _) = launches()
        assert ("Li8ELb%dELi" % over) in reduce and ("Li8ELb%dEEE" % over) in scatter, (reduce, scatter)
        assert block[0] == (512 if over or es == 4 else 256), block
""")


def test_alltoalls_that_nearly_fill_the_cache_are_streamed(recorded):  # noqa: F811
    """From 112 MiB of sources on, without a gap where the cache ends (second template argument)."""
    recorded("""
ok(lib.nvshmemx_amd_init(4, 256 << 20))
a, b = lib.nvshmem_malloc(96 << 20), lib.nvshmem_malloc(96 << 20)
for mib, streamed in ((28, 0), (29, 1), (63, 1), (64, 1), (65, 1)):
    launches()
    ok(lib.nvshmemx_alltoallmem_on_stream(0, b, a, mib << 18, None))
    (kernel, _, _, _, _), = launches()
    assert "ILi1ELb%dELb0E" % streamed in kernel, (mib, kernel)
""")


def test_large_teams_fold_into_one_member_and_broadcast(recorded):  # noqa: F811
    """From 16 members and 96 MiB of sources in all on: two launches, the second from the first member's destination."""
    recorded("""
for npes, mib, two in ((15, 8, 0), (16, 5, 0), (16, 6, 1), (16, 32, 1), (32, 3, 1), (33, 2, 0), (64, 2, 1)):
    ok(lib.nvshmemx_amd_init(npes, 80 << 20))
    a, b = lib.nvshmem_malloc(32 << 20), lib.nvshmem_malloc(32 << 20)
    launches()
    ok(_lib.typed_coll(lib, "nvshmemx_float_sum_reduce_on_stream", True)(0, b, a, mib << 18, None))
    names = [l[0] for l in launches()]
    assert len(names) == 1 + two, (npes, mib, names)
    assert not two or ("reduce_root_kernel" in names[0] and "segment_copy_kernelILi2" in names[1]), names
    lib.nvshmem_finalize()
""")


def test_sources_that_a_program_keeps_in_the_cache_stay_with_the_fused_reduction(recorded):  # noqa: F811
    """With a larger NVSHMEM_AMD_CACHEABLE_SOURCE_BYTES large teams take two steps from 3/8 of that on, as their sources are
    streamed from there; with a smaller one still from 96 MiB.  A threshold of its own wins."""
    code = """
ok(lib.nvshmemx_amd_init(16, 80 << 20))
a, b = lib.nvshmem_malloc(32 << 20), lib.nvshmem_malloc(32 << 20)
for mib, two in %s:
    launches()
    ok(_lib.typed_coll(lib, "nvshmemx_float_sum_reduce_on_stream", True)(0, b, a, mib << 18, None))
    names = [l[0] for l in launches()]
    assert len(names) == 1 + two and ("reduce_root_kernel" in names[0]) == bool(two), (mib, names)
"""
    cacheable = {"NVSHMEM_AMD_CACHEABLE_SOURCE_BYTES": str(1 << 30)}
    recorded(code % "((6, 0), (16, 0), (23, 0), (24, 1))", **cacheable)
    recorded(code % "((1, 0), (5, 0), (6, 1))", NVSHMEM_AMD_CACHEABLE_SOURCE_BYTES="0")
    recorded(code % "((7, 0), (8, 1), (16, 1))", NVSHMEM_AMD_TWO_STEP_REDUCE_BYTES=str(128 << 20), **cacheable)


def test_streamed_sources_on_another_offset_share_their_lines(recorded):  # noqa: F811
    """Two members: the gather kernel whose lanes at a tile's ends load cacheable (fifth template argument), as long as the
    cache could hold the sources.  A whole number of lines apart there are none to share."""
    recorded("""
ok(lib.nvshmemx_amd_init(2, 512 << 20))
a, b = lib.nvshmem_malloc(160 << 20), lib.nvshmem_malloc(160 << 20)
for mib, offset, kernel in ((48, 4, "Li0ELb0ELb0E"), (49, 0, "Li0ELb1ELb0E"), (49, 128, "Li0ELb1ELb0E"), (49, 4, "Li0ELb1ELb1E"),
                            (49, 16, "Li0ELb1ELb1E"), (128, 4, "Li0ELb1ELb1E"), (129, 4, "Li0ELb1ELb0E")):
    launches()
    ok(_lib.typed_coll(lib, "nvshmemx_float_sum_reduce_on_stream", True)(0, b, a + offset, mib << 18, None))
    (name, _, _, _, _), = launches()
    assert "reduce_gather_kernel" in name and kernel in name, (mib, offset, name)
""")


def test_streamed_sources_of_large_teams_share_the_kernels_of_any_team_size(recorded):  # noqa: F811
    """A program that switches the two-step form off: the staged kernel that reads the team size, two members to a wavefront."""
    recorded("""
for npes, mib in ((16, 7), (32, 4)):
    ok(lib.nvshmemx_amd_init(npes, 80 << 20))
    a, b = lib.nvshmem_malloc(32 << 20), lib.nvshmem_malloc(32 << 20)
    launches()
    for per_pe in (mib, 5 if npes == 16 else 2):
        ok(_lib.typed_coll(lib, "nvshmemx_float_sum_reduce_on_stream", True)(0, b, a, per_pe << 18, None))
    (streamed, _, _, block, _), (cached, _, _, _, _) = launches()
    assert "reduce_vector_kernelIfLi5ELi0ELb1ELi1ELi2E" in streamed and block[0] == 32 * npes, (streamed, block)
    assert "reduce_vector_kernelIfLi5ELi%dELb0E" % npes in cached, cached
    lib.nvshmem_finalize()
""", NVSHMEM_AMD_TWO_STEP_REDUCE_MEMBERS="0")
