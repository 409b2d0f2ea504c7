// Host-launched collectives for logical PEs on one MI355X: one grid-wide kernel per call serves
// every PE of the team - and, when the handle names a family of disjoint teams (the rows of a 2-D
// split), every team of the family: grid.z indexes the team, whose <start, stride, size> the kernel
// reads from the device copy of the team table.
//
// Reference counterparts: the on-stream launchers src/host/stream/coll/{rdxn/reduce_common.cuh:29-68,
// fcollect/fcollect.cu:20-65, alltoall/alltoall.cu:18-40} start one block per PE that runs the
// device templates coll/reduce.cuh:1592-1674, coll/fcollect.cuh:331-344, coll/alltoall.cuh:122-143
// and meets the other PEs in a flag barrier.  Here all PEs share one HBM, so a collective is a
// single streaming pass: every source byte is read once, every destination byte written once, and
// the kernel boundary is the barrier.
//
//   reduce    dest@q[k] = fold_{p = 0..n-1, in that order} src@p[k]      for every PE q
//   fcollect  dest@q[p*nelems + k] = src@p[k]                            for every PE q
//   alltoall  dest@q[p*nelems + k] = src@p[q*nelems + k]
//   broadcast dest@q[k] = src@root[k]                                    for every PE q
//   reducescatter  dest@q[k] = fold_{p = 0..n-1} src@p[q*nreduce + k]
//
// Reference counterparts of the last two: src/host/coll/broadcast/broadcast.cpp with
// coll/broadcast.cuh:276-337, src/host/coll/reducescatter/reducescatter_on_stream.cpp with
// coll/reducescatter.cuh:36-90.
#include <cstdio>

#include "nvshmem.h"
#include "launch.hpp"
#include "runtime.hpp"

namespace nvshmem_amd {
namespace {

// Tunables (compile time).  Defaults are the values measured best on MI355X.
#ifndef NVSHMEM_AMD_REDUCE_VPT /* vectors a thread of the fused reduce loads per tile */
#define NVSHMEM_AMD_REDUCE_VPT 1
#endif
#ifndef NVSHMEM_AMD_REDUCE_VPT_NARROW /* the same for 1- and 2-byte elements on the compile-time team sizes 8 and 16 */
#define NVSHMEM_AMD_REDUCE_VPT_NARROW 1
#endif
/* Members per wavefront of the fused reduce on teams of 8 and on cached sources of 16, for 1- and 2-byte
 * elements (NARROW) and for wider ones (WIDE).  Narrow elements fold twice to four times as many elements
 * per byte, and a block has nothing in flight while it folds: with two members per wavefront the blocks
 * are half as large and twice as many share a compute unit, so more of them are in their load or store
 * phase at any time (16 members of bf16, cached sources of 70 MB in all: 22.2 us, 24.3 with one).  Streamed sources of 8
 * members take one all the same: two loads of a wavefront, back to back, cost more than that gains (8 members of bf16,
 * 100 | 200 | 400 | 1600 MB: 35.5 | 66.9 | 132.3 | 525 us with two members, 34.5 | 65.2 | 128.4 | 503 with one; four 36.8 | 69.8 |
 * 137.6 | 548).  4- and 8-byte elements lose 5 % with two members per wavefront and 11 % with four. */
#ifndef NVSHMEM_AMD_REDUCE_NARROW_MPW
#define NVSHMEM_AMD_REDUCE_NARROW_MPW 2
#endif
#ifndef NVSHMEM_AMD_REDUCE_WIDE_MPW
#define NVSHMEM_AMD_REDUCE_WIDE_MPW 1
#endif
#ifndef NVSHMEM_AMD_COLL_NT /* non-temporal loads allowed */
#define NVSHMEM_AMD_COLL_NT 1
#endif
/* Sources of up to Runtime::cacheable_source_bytes (all PEs together, 256 MiB unless the environment
 * says otherwise) are loaded with the default, cacheable policy: they fit the 256 MiB Infinity
 * Cache, so a source that is sent again is served from it (measured +30 % on
 * the 1M-element reduce, +20..45 % on 256 MiB collectives).  Larger sources are streamed with
 * non-temporal loads (+5 % at 2 GiB).  Stores always stream.
 *
 * Reductions stream from 3/8 of that on (96 MiB, streamed_reduction).  A streamed load is served from the Infinity
 * Cache where the line is there - a source that was just produced - but brings none into it, so it does not push out
 * what others have written there and not yet to memory.  us cached / streamed loads, fp32 normal data, sources in all of 110 | 160 |
 * 200 MB | 256 MiB (16 members cached on the fused kernel, streamed in two steps):
 *  - three sets of buffers in turn, each source filled in front of its call, both kernels: allreduce on 4 members 57.9 / 55.2 | 86.4 /
 *    75.1 | 105.6 / 90.6 | 118.8 / 117.7, 8 members 73.2 / 70.1 | 104.8 / 87.0 | 122.9 / 102.4 | 133.2 / 132.2, 16 members 88.5 / 80.8 |
 *    119.3 / 103.2 | 143.4 / 123.6 | 146.4 / 152.2; reducescatter on 8 members 54.1 / 52.1 | 68.6 / 67.9 | 80.4 / 79.5 | 104.6 / 100.7.
 *  - in turn without the fills: allreduce on 4 members 39.1 / 37.8 | 54.0 / 52.9 | 67.7 / 65.7 | 89.1 / 85.9, 8 members 43.7 / 42.7 |
 *    58.4 / 54.5 | 72.2 / 67.4 | 97.4 / 88.0; reducescatter on 8 members, 128 MiB | 200 MB | 256 MiB, 30.2 / 27.3 | 43.7 / 37.6 | 56.3 / 49.5.
 *  - below 96 MiB sources that are in use in turn are still there: of 64 MB allreduce 19.2 / 23.7, reducescatter 11.7 / 12.6.
 * What loses:
 *  - A source that is reduced again as it is, with nothing in between (a sum and then a maximum of one buffer): 128 MiB | 200 MB | 256
 *    MiB on 4 members 37.9 / 43.6 | 55.2 / 65.6 | 73.5 / 85.5, 8 members 43.0 / 47.3 | 60.6 / 68.7 | 79.0 / 89.0, 16 members 39.9 / 45.3 |
 *    57.9 / 63.4 | 76.5 / 83.3, 32 members 39.6 / 48.7 | 57.7 / 68.5 | 76.6 / 88.8; reducescatter on 8 members 25.8 / 25.7 | 35.8 / 37.4 |
 *    48.9 / 50.1.  Buffers of zeros, which the cache serves faster, lose up to 40 % (8 members 36.4 / 43.4 and 67.2 / 84.6, 32 34.5 / 48.2).
 *  - ONE source that is filled again in front of each call on 8 and 16 members (both kernels less the fill alone): 8 members 51.1 /
 *    55.8 | 60.2 / 66.4 | 68.8 / 73.9 | 87.8 / 86.2, 16 members 39.5 / 41.5 | 50.1 / 57.8 | 64.5 / 69.5 | 81.6 / 87.2; 4 members gain, 41.7 /
 *    39.7 | 58.1 / 51.5 | 66.9 / 61.7 | 86.7 / 81.0.
 *  - Sources on another offset in a line near the cache's size: stream_load_astride.
 * A larger cacheable_source_bytes is for programs of these kinds.  (A quarter kept, as an alltoall's: in turn without fills 86.1
 * instead of 88.0, 8 members of 256 MiB; with them 162 instead of 132.) */

// (any byte alignment: one global_load_dwordx4 either way)
template <bool NTL>
__device__ __forceinline__ nvshmemi_v4u stream_load(const char *p) {
    if (NTL && NVSHMEM_AMD_COLL_NT)
        return __builtin_nontemporal_load(reinterpret_cast<const nvshmemi_v4u_unaligned *>(p));
    return *reinterpret_cast<const nvshmemi_v4u_unaligned *>(p);
}
// A streamed load of a wavefront whose KiB does not start on a line of its own: the lines at its ends, which the wavefronts
// on either side read too, possibly on another XCD, are brought into the caches (`shared`: the lanes on them), as
// streamed ones come from memory twice.  us cached / streamed / so, allreduce, source on another offset, 110 | 160 | 200 MB | 256 MiB of
// sources in all, fp32 normal data: three sets in turn, each filled in front of its call (both kernels), 2 members 51.9 / 58.5 / 52.6 |
// 78.0 / 82.3 / 73.8 | 93.6 / 101.3 / 92.4 | 115.6 / 134.4 / 127.8, 4 members 60.7 / 68.5 / 60.2 | 91.1 / 93.5 / 80.5 | 108.5 / 110.3 /
// 101.2 | 125.4 / 145.2 / 149.9, 8 members 71.4 / 77.4 / 67.8 | 106.1 / 101.1 / 92.7 | 124.4 / 122.5 / 122.7 | 139.2 / 161.0 / 167.6: at
// the cache's own size it is the whole of streaming that loses.  In turn without fills 8 members 42.9 / 42.5 / 41.5 | 61.7 / 58.4 /
// 58.6 | 80.5 / 76.5 / 75.2 | 110.0 / 99.7 / 98.3; reduced again as it is 36.1 / 45.6 / 43.8 | 51.0 / 60.5 / 58.5 | 65.2 / 78.4 / 74.9 |
// 88.0 / 106.1 / 106.1.  (The empty statements keep the compiler from making one plain load of the two.)
__device__ __forceinline__ nvshmemi_v4u stream_load_astride(const char *p, bool shared) {
    nvshmemi_v4u v;
    if (shared) {
        asm volatile("");
        v = stream_load<false>(p);
        asm volatile("");
    } else {
        v = stream_load<true>(p);
    }
    return v;
}
// Blocks go to the eight XCDs in turn, and so would tiles that share lines of a source (it starts on another offset in
// a line than the destination, on whose lines tiles are cut): each of these lines would come into two L2s.  The first
// `dealt` blocks, a multiple of 8 * kDealtTiles, take tiles so that kDealtTiles consecutive ones share an XCD.  us in order /
// dealt by 2 | 4 | 8 | 16, allreduce, sources on another offset: 8 members fp32 60 MB of sources in all 19.2 / 19.6 | 18.4 | 18.9 |
// 18.2, 110 MB streamed 39.7 / 38.5 | 37.9 | 38.9 | 40.1, 420 MB 141.7 / 142.8 | 136.6 | 140.3 | 146.9; 2 members 110 MB 37.7 / 36.7 |
// 36.1 | 36.4 | 36.2, 420 MB 134.7 / 131.7 | 129.0 | 131.6 | 131.8.  Where no line is shared it only widens what is read at a time
// (8 members, 420 MB aligned: 132.4 in order, by 8 138.4).  Small ones, in order / dealt by 4, three sets in turn in a graph: 2 to
// 16 members the same below 1 MiB per PE; 1 MiB 4 members fp32 2.80 / 2.33, 8 bf16 4.73 / 4.05, 16 bf16 8.88 / 8.34, 2 bf16 2.55 /
// 2.57; 4 MiB 8 members fp32 13.3 / 11.9, 16 members 22.3 / 22.6, bf16 21.8 / 23.0, the most that loses (sent again as it is 21.8 / 21.5).
constexpr unsigned kDealtTiles = 4;
__device__ __forceinline__ unsigned dealt_tile(unsigned block, unsigned dealt) {
    constexpr unsigned kGroup = 8 * kDealtTiles;
    return block < dealt ? block / kGroup * kGroup + block % 8 * kDealtTiles + block / 8 % kDealtTiles : block;
}
static uint32_t dealt_blocks(uint64_t dst_off, uint64_t src_off, uint64_t blocks) {
    return (dst_off - src_off) % 128 ? (uint32_t)(blocks / (8 * kDealtTiles) * (8 * kDealtTiles)) : 0;
}
// How a kernel's result stores treat the caches.  Both forms write through (nothing here reads its output back): the
// line leaves the L2 at once instead of queuing behind its eviction of streaming lines, and a write-only stream
// reaches 7.2 TB/s against 6.3 TB/s with nt alone.  Which of the two wins depends on the kernel's mix (measured on
// MI355X, random data, against nt): sc1 nt +4.5 % for the 8-member allreduce, +5..10 % for fcollect and broadcast,
// +1..3 % for alltoall and the gather allreduce; plain sc1 +5 % for the reducescatter, whose one store per eight loads
// gains nothing from nt.
enum { kStoreThrough = 1 /* sc1 */, kStoreThroughStream = 2 /* sc1 nt */ };
#ifndef NVSHMEM_AMD_STORE_ALLTOALL
#define NVSHMEM_AMD_STORE_ALLTOALL kStoreThroughStream
#endif
#ifndef NVSHMEM_AMD_STORE_REPLICATE /* fcollect and broadcast, one wavefront storing to every member */
#define NVSHMEM_AMD_STORE_REPLICATE kStoreThroughStream
#endif
#ifndef NVSHMEM_AMD_STORE_REDUCE
#define NVSHMEM_AMD_STORE_REDUCE kStoreThroughStream
#endif
#ifndef NVSHMEM_AMD_STORE_REDUCESCATTER
#define NVSHMEM_AMD_STORE_REDUCESCATTER kStoreThrough
#endif
// The team a block serves: among the kernel's arguments when the handle names one team, else row `group` of the
// device's team table (which costs a load that everything else waits for).
struct team_arg_t {
    nvshmemi_amd_team_view_t one;
    const nvshmemi_amd_team_view_t *table;  // null: one
};
static team_arg_t team_arg(const TeamLaunch &tl) { return {tl.first, tl.ngroups > 1 ? tl.groups : nullptr}; }
__device__ __forceinline__ nvshmemi_amd_team_view_t team_of(const team_arg_t &t, unsigned group) {
    return t.table ? t.table[group] : t.one;
}

// The asm forms end in s_nop 1: the compiler does not know the statement is a store of more than 8 bytes
// and would not keep the wait state this GPU needs before the data registers are written again.
template <int STORE>
__device__ __forceinline__ void stream_store(char *p, nvshmemi_v4u v) {
    if (STORE == kStoreThrough)
        asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"(p), "v"(v) : "memory");
    else
        asm volatile("global_store_dwordx4 %0, %1, off sc1 nt\n\ts_nop 1" : : "v"(p), "v"(v) : "memory");
}
// The same at p + off, p the same for all lanes: the address stays a scalar base and a 32-bit offset per lane.  (The
// s_nop in front: a vector instruction that wrote the base - the compiler may have moved it out of a vector
// register - must be five wait states away.)
template <int STORE>
__device__ __forceinline__ void stream_store_at(char *p, unsigned off, nvshmemi_v4u v) {
    if (STORE == kStoreThrough)
        asm volatile("s_nop 4\n\tglobal_store_dwordx4 %0, %1, %2 sc1\n\ts_nop 1" : : "v"(off), "v"(v), "s"(p) : "memory");
    else
        asm volatile("s_nop 4\n\tglobal_store_dwordx4 %0, %1, %2 sc1 nt\n\ts_nop 1" : : "v"(off), "v"(v), "s"(p) : "memory");
}

// ---------------------------------------------------------------------------------------------
// Segment copy: fcollect and alltoall are sets of contiguous (source, destination) segments, a broadcast is one.
// grid.y (alltoall: grid.y and grid.z) indexes the segment, grid.x the tile inside it.  A block is ONE wavefront that
// moves ONE aligned 1 KiB piece (64 lanes x 16 bytes): on MI355X this shape measured fastest by a clear
// margin (6.7-6.8 TB/s for alltoall, against 6.0 TB/s with 256-thread blocks and 8 KiB tiles and
// 4.0 TB/s with 32 KiB tiles), because the blocks in flight then cover a narrow, moving window of
// addresses.  The destination is written with aligned vectors only: block 0 of a segment copies
// the byte head in front of the first aligned destination vector and the byte tail behind the
// last one.
//
// fcollect and broadcast store the piece to every member, in one of two ways:
//  - back to back, while the whole grid is in flight at once.  Small messages are latency: with the stores of a loop
//    that waits for each before the next, every destination costs a quarter of a microsecond (64 bytes to 64 KiB per
//    member, replayed from a graph: fcollect to 8 / 16 members 3.4-4.5 / 5.4-6.9 us one by one, 1.9-2.9 / 2.0-4.1 back to
//    back, broadcast of up to 64 KiB to 8 3.1-3.9 and 1.8-2.1);
//  - PACED, one destination after the other, each store acknowledged before the next is issued, in larger grids.
//    They are bound by how the memory system takes writes, and that favours few write fronts: blocks that start
//    together then write to one destination at a time instead of all 8 or 16 (broadcast of 32 MiB to 8: 47.4 us back
//    to back, 42.8 paced), and the fewer wavefronts take part, the narrower each front.  So the launch also limits
//    how many a compute unit holds (paced_lds_bytes).
// A CHUNKED fcollect (streamed sources, 16 members and more) is paced with two destinations to a wavefront: the grid
// walks a chunk of tiles once per pair of destinations, re-reading it from the cache, before it goes on to the next.
// The pieces in flight then feed a few write fronts however many members there are (chunked_copy).
// ---------------------------------------------------------------------------------------------

enum { kModeFcollect = 0, kModeAlltoall = 1, kModeBroadcast = 2 };
// Below this length of a segment the edge bytes are stored in front of the vectors, which mostly lie in the same lines;
// beyond, behind them, so that the vectors of block 0 are on their way no later than those of the other blocks.  us
// first / last: broadcast to 8 of 64 bytes on an odd address 2.0 / 2.2, of 800 2.2 / 2.1; alltoall on 16 PEs of 200 bytes
// 2.4 / 2.5, of 1021 2.6 / 2.3, of 16372 4.4 / 3.7.
constexpr unsigned kEdgesFirstBytes = 512;

struct segment_args_t {
    char *base;
    uint64_t slice_bytes;
    team_arg_t team;
    uint64_t dst_off, src_off, seg_bytes;
    uint32_t root;
    uint32_t members;                  // of the handle's largest team (gridDim would cost the host 0.6 us a launch: host_rma.hip)
    uint16_t part_shift, chunk_shift;  // chunked walk: 2^part_shift groups of destinations, chunks of 2^chunk_shift tiles
    bool astride;                      // streamed alltoall: lanes at the ends of a piece load cacheable (segment_collective)
};

template <int MODE, bool NTL, bool PACED, int STORE, bool CHUNKED = false>
__global__ __launch_bounds__(64) void segment_copy_kernel(segment_args_t a) {
    // this block's team: members are the PEs start + i*stride, i < size
    unsigned p = MODE == kModeAlltoall ? blockIdx.z : blockIdx.y, group = MODE == kModeAlltoall ? 0 : blockIdx.z;
    if (MODE == kModeAlltoall && a.team.table) {
        group = p / a.members;
        p -= group * a.members;
    }
    const nvshmemi_amd_team_view_t g = team_of(a.team, group);
    const unsigned npes = (unsigned)g.size;
    char *const base = a.base + (uint64_t)(unsigned)g.start * a.slice_bytes;
    const uint64_t rep_stride = (uint64_t)(unsigned)g.stride * a.slice_bytes;  // from one member to the next
    const char *src;
    char *dst;
    unsigned nrep = npes;
    if (MODE == kModeFcollect) {
        // segment p: member p's source -> slot p of every member's destination
        if (p >= npes) return;
        src = base + p * rep_stride + a.src_off;
        dst = base + a.dst_off + p * a.seg_bytes;
    } else if (MODE == kModeBroadcast) {
        // one segment: the root's source -> every member's destination
        src = base + a.root * rep_stride + a.src_off;
        dst = base + a.dst_off;
    } else {
        // segment (p, q): block q of member p's source -> slot p of member q's destination
        const unsigned q = blockIdx.y;
        if (p >= npes || q >= npes) return;
        src = base + p * rep_stride + a.src_off + q * a.seg_bytes;
        dst = base + q * rep_stride + a.dst_off + p * a.seg_bytes;
        nrep = 1;
    }
    unsigned tile = blockIdx.x;
    if (CHUNKED) {
        const unsigned part = (tile >> a.chunk_shift) & ((1u << a.part_shift) - 1);
        tile = (tile & ((1u << a.chunk_shift) - 1)) + (tile >> (a.chunk_shift + a.part_shift) << a.chunk_shift);
        const unsigned per = (npes + (1u << a.part_shift) - 1) >> a.part_shift, r0 = part * per;
        if (r0 >= npes) return;  // a team smaller than the grid's largest: nothing left for this group
        nrep = npes - r0 < per ? npes - r0 : per;
        dst += r0 * rep_stride;
    }
    const unsigned lane = threadIdx.x;
    unsigned head = (unsigned)(-(uintptr_t)dst) & 15;
    if (head > a.seg_bytes) head = (unsigned)a.seg_bytes;
    const uint64_t nvec = (a.seg_bytes - head) / 16;
    // tiles are cut on absolute 1 KiB boundaries of the destination: `lead` vector slots of tile 0
    // lie in front of the segment
    const unsigned lead = (unsigned)((uintptr_t)(dst + head) >> 4) & 63;
    const int64_t v0 = (int64_t)tile * 64 - lead, left = (int64_t)nvec - v0;
    const bool edges = tile == 0;  // this block also moves the bytes around the vectors
    if (left <= 0 && !edges) return;
    // this lane's vector, as an unsigned index: slots in front of the segment wrap and are skipped like those behind it
    const unsigned first = edges ? lead : 0, end = left < 64 ? (unsigned)left : 64;
    const bool body = lane - first < end - first;
    nvshmemi_v4u v = {};
    if (body) {
        const char *const from = src + head + 16 * v0 + 16 * lane;
        if (MODE == kModeAlltoall && NTL && a.astride) v = stream_load_astride(from, lane - 8 >= 48);
        else v = stream_load<NTL>(from);
    }
    // at most 15 + 15 bytes, lane k the k-th of them, every second destination on either half of the lanes; they are
    // loaded beside the vectors
    const unsigned k = lane & 31;
    const bool edge = edges && k < head + ((unsigned)(a.seg_bytes - head) & 15);
    const uint64_t pos = k < head ? k : nvec * 16 + k;
    unsigned b = 0;
    if (edge) b = (unsigned char)src[pos];
    // The wait for both loads belongs here, once: left to the compiler it stands in front of every group of stores below,
    // where it also waits for the stores before (fcollect to 16 / 64 members of 64 bytes 2.3 / 5.5 us, like this 2.0 / 3.6).
    // An alltoall stores once, and its edge bytes do better behind the vectors' acknowledgement (16 PEs, 65533 bytes: 6.7
    // us against 6.85); a paced copy waits in any case, and with streamed loads it loses 10 % by the wait out here
    // (broadcast of 512 MiB to 8 734 us, 807 so; fcollect of 16 x 32 MiB 1446 and 1629).
    if (MODE != kModeAlltoall && !PACED) asm volatile("" : "+v"(v), "+v"(b));
    auto store_edges = [&]() {
        if (!edge) return;
        const unsigned half = lane >> 5;
        char *to = dst + half * rep_stride + pos;
#pragma nounroll
        for (unsigned r = 0; r < nrep; r += 2, to += 2 * rep_stride)
            if (r + half < nrep) *to = (char)b;
    };
    const bool edges_first = a.seg_bytes < kEdgesFirstBytes;
    if (edges_first) store_edges();
    char *d = dst + head + 16 * v0;
    auto store = [&](char *to) { stream_store_at<STORE>(to, 16 * lane, v); };
    if (body) {
        unsigned n = nrep;
        if (MODE == kModeAlltoall) {
            store(d);
        } else if (PACED) {
            store(d);
            while (--n) {
                d += rep_stride;
                nvshmemi_amd_wait_vm();
                store(d);
            }
        } else {
            for (; n >= 8; n -= 8, d += 8 * rep_stride) {
#pragma unroll
                for (int r = 0; r < 8; ++r) store(d + r * rep_stride);
            }
            if (n >= 4) {
#pragma unroll
                for (int r = 0; r < 4; ++r) store(d + r * rep_stride);
                n -= 4, d += 4 * rep_stride;
            }
            for (; n; --n, d += rep_stride) store(d);
        }
    }
    if (!edges_first) store_edges();
}

// ---------------------------------------------------------------------------------------------
// Fused reduce, LDS staged.  A block owns a tile of 64 16-byte vectors of the element range and has one
// wavefront per MPW members of the team, so a wavefront streams one aligned 1 KiB piece of a member's
// source per load.  Thread (w, i) loads vector i of the tile from members w*MPW ... w*MPW + MPW-1 into
// LDS - one load per lane and member, like a plain copy, which HBM serves measurably faster than one
// lane gathering the same vector from every PE.  After a barrier the tile's elements are folded out of
// LDS in PE order 0..n-1, one element per thread, and thread (w, i) stores result vector i into the
// destinations of its members.
// An element is read (by the loads of this block) before this block writes it and no other block
// touches it, so dest == src (in place) needs no further staging.
// ---------------------------------------------------------------------------------------------
// NPES > 0 fixes the team size at compile time (fold fully unrolled); NPES == 0 takes it from the team
// table, the block being sized for the largest team of the handle.
// fold_next: one step of the fold, in the allreduce's operand order or (SCATTER) the reducescatter's.
template <typename T, int OP, bool SCATTER>
__device__ __forceinline__ T fold_next(int p, T acc, T x) {
    return SCATTER ? nvshmemi_amd_reduce_op<T, OP>(acc, x) : nvshmemi_amd_fold_step<T, OP>(p, acc, x);
}

// What a reduction moves, the same for every member (the slices lie a multiple of 2 MiB apart, so an offset has the
// same alignment in all of them): whole vectors from the first 16-byte boundary of the destination on, and the
// elements in front of and behind them, fewer than 16 bytes on either side.  Stores are aligned that way whatever
// the buffers are; a source on another offset is read with unaligned vector loads, which cost 3-4 % here (allreduce of
// 8 x 25 MiB bf16: 73 us with both buffers on the same offset, aligned or not, 76 with different ones; an
// element per lane and load takes 155 and 148 us).
struct reduce_shape_t {
    uint64_t dst, src;   // byte offsets of the destination and the source in a slice
    uint64_t nvec;       // whole vectors
    uint32_t head, tail; // elements in front of and behind them
    uint32_t lead;       // the first vector's place in its aligned 1 KiB of the destination
    uint32_t dealt;      // blocks whose tiles are dealt to the XCDs (dealt_tile)
    bool astride;        // streamed loads share the lines at a tile's ends (stream_load_astride)
};
template <typename T>
reduce_shape_t reduce_shape(const Runtime &rt, uint64_t dst_off, uint64_t src_off, uint64_t nelems) {
    const uint64_t at = (uint64_t)(uintptr_t)rt.base + dst_off;
    uint64_t head = (-at & 15) / sizeof(T);
    if (head > nelems) head = nelems;
    const uint64_t nvec = (nelems - head) / (16 / sizeof(T));
    return {dst_off, src_off, nvec, (uint32_t)head, (uint32_t)(nelems - head - nvec * (16 / sizeof(T))),
            (uint32_t)((at + head * sizeof(T)) >> 4 & 63), 0, false};
}
// The elements around the vectors, one per thread of the calling block's first wavefront.
template <typename T, int OP, bool SCATTER>
__device__ __forceinline__ void reduce_edges(char *dst, const char *src, const reduce_shape_t &s, uint64_t pe_stride,
                                             int npes, int copies) {
    if (threadIdx.x >= s.head + s.tail) return;
    const uint64_t k = threadIdx.x < s.head ? threadIdx.x : s.nvec * (16 / sizeof(T)) + threadIdx.x;
    const T *from = reinterpret_cast<const T *>(src) + k;
    const uint64_t es = pe_stride / sizeof(T);
    T acc = from[0];
    constexpr int kBatch = 8;  // loads in flight (beyond the last member: that one again)
    for (int p0 = 1; p0 < npes; p0 += kBatch) {
        T x[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) x[j] = from[(uint64_t)(p0 + j < npes ? p0 + j : npes - 1) * es];
#pragma unroll
        for (int j = 0; j < kBatch; ++j)
            if (p0 + j < npes) acc = fold_next<T, OP, SCATTER>(p0 + j, acc, x[j]);
    }
    for (int p = 0; p < copies; ++p) reinterpret_cast<T *>(dst + (uint64_t)p * pe_stride)[k] = acc;
}

template <typename T, int OP, int NPES, bool NTL, int VPT = NVSHMEM_AMD_REDUCE_VPT, int MPW = 1>
__global__ __launch_bounds__(NPES ? NPES / MPW * 64 : 1024) void reduce_vector_kernel(char *base, uint64_t slice_bytes,
                                                             const nvshmemi_amd_team_view_t *groups,
                                                             reduce_shape_t s) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    constexpr int VEC = 16 / sizeof(T);
    // this block's team; with NPES > 0 the host has checked that every team has NPES members
    const nvshmemi_amd_team_view_t g = groups[blockIdx.z];
    const int npes = NPES ? NPES : g.size;
    base += (uint64_t)g.start * slice_bytes;
    constexpr uint32_t lane_shift = 6;  // a wavefront's 64 lanes move one aligned 1 KiB piece of a member
    constexpr unsigned lanes = 1u << lane_shift;
    // a wavefront serves MPW consecutive members (more than one only with a compile-time team size)
    // (the wavefront's index as a scalar: the members' base addresses then stay in scalar registers)
    const unsigned pe0 = (unsigned)__builtin_amdgcn_readfirstlane(threadIdx.x >> lane_shift) * MPW,
                   i = threadIdx.x & (lanes - 1);
    char *const dst = base + s.dst + s.head * sizeof(T);
    const char *const src = base + s.src + s.head * sizeof(T);
    // tiles are cut on absolute (16 * lanes)-byte boundaries of the destination, so a wavefront's
    // access is one aligned 1 KiB piece whatever the buffer's own alignment: `lead` vector slots of
    // the first tile lie in front of the buffer
    const uint64_t pe_stride = (uint64_t)g.stride * slice_bytes;  // from one member to the next
    // the block is sized for the largest team of the handle: lanes of members a team does not have idle
    auto member = [&](int m) { return NPES ? true : (int)pe0 + m < npes; };
    // a tile is VPT pieces of `lanes` vectors per PE: thread (pe, i) loads vector i of each piece
    constexpr unsigned tile_vecs = (unsigned)VPT << lane_shift;
    nvshmemi_v4u *stage = reinterpret_cast<nvshmemi_v4u *>(lds);           // [npes][tile_vecs]
    nvshmemi_v4u *result = stage + (size_t)npes * tile_vecs;               // [tile_vecs]
    // the unit of the fold: a 4-byte word (EPW elements) for 1- and 2-byte elements, else one element
    constexpr int EPW = sizeof(T) < 4 ? 4 / (int)sizeof(T) : 1;
    struct alignas(sizeof(T) * EPW) word_t {
        T e[EPW];
    };
    const word_t *stage_w = reinterpret_cast<const word_t *>(stage);
    word_t *result_w = reinterpret_cast<word_t *>(result);
    constexpr unsigned tile_words = tile_vecs * VEC / EPW;

    // indices in front of the buffer wrap to huge values and are skipped like those behind it
    const uint64_t v0 = (uint64_t)dealt_tile(blockIdx.x, s.dealt) * tile_vecs + i - s.lead;
    auto fetch = [&](auto load) {
#pragma unroll
        for (int u = 0; u < VPT; ++u) {
            const uint64_t v = v0 + ((uint64_t)u << lane_shift);
            if (v < s.nvec) {
#pragma unroll
                for (int m = 0; m < MPW; ++m)
                    if (member(m)) stage[(pe0 + m) * tile_vecs + ((unsigned)u << lane_shift) + i] =
                        load(src + (uint64_t)(pe0 + m) * pe_stride + 16 * v);
            }
        }
    };
    // (stream_load_astride has the figures.  Sources beyond the Infinity Cache lose more by what this pushes out of it than they
    // gain: 8 members, 300 MB just written 104 / 113 us, 420 MB 128 / 142, in turn 136.4 / 134.3.)
    if (NTL && s.astride) fetch([i](const char *p) { return stream_load_astride(p, i - 8 >= 48); });
    else fetch([](const char *p) { return stream_load<NTL>(p); });
    __syncthreads();
    // a thread folds one 4-byte word of the tile at a time - one element of 4 or 8 bytes, or the 2 or 4
    // narrower elements that share the word, each folded on its own in member order - so that a tile of
    // 1- or 2-byte elements costs as many LDS instructions as one of 4-byte elements
    for (unsigned w = threadIdx.x; w < tile_words; w += blockDim.x) {
        typedef nvshmemi_amd_fold_form<T, OP> form;
        const word_t first = stage_w[w];
        typename form::acc_t acc[EPW];
#pragma unroll
        for (int j = 0; j < EPW; ++j) acc[j] = form::lift(first.e[j]);
        if (NPES) {
#pragma unroll
            for (int p = 1; p < NPES; ++p) {
                const word_t x = stage_w[(size_t)p * tile_words + w];
#pragma unroll
                for (int j = 0; j < EPW; ++j) acc[j] = form::step(p, acc[j], x.e[j]);
            }
        } else {
            // eight members' values fetched from LDS before they are folded, in member order
            int p = 1;
            for (; p + 8 <= npes; p += 8) {
                word_t x[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) x[k] = stage_w[(size_t)(p + k) * tile_words + w];
#pragma unroll
                for (int k = 0; k < 8; ++k)
#pragma unroll
                    for (int j = 0; j < EPW; ++j) acc[j] = form::step(p + k, acc[j], x[k].e[j]);
            }
            for (; p < npes; ++p) {
                const word_t x = stage_w[(size_t)p * tile_words + w];
#pragma unroll
                for (int j = 0; j < EPW; ++j) acc[j] = form::step(p, acc[j], x.e[j]);
            }
        }
        word_t out;
#pragma unroll
        for (int j = 0; j < EPW; ++j) out.e[j] = form::lower(acc[j]);
        result_w[w] = out;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < VPT; ++u) {
        const uint64_t v = v0 + ((uint64_t)u << lane_shift);
        const nvshmemi_v4u r = result[((unsigned)u << lane_shift) + i];
        if (v < s.nvec) {
#pragma unroll
            for (int m = 0; m < MPW; ++m)
                if (member(m)) stream_store<NVSHMEM_AMD_STORE_REDUCE>(dst + (uint64_t)(pe0 + m) * pe_stride + 16 * v, r);
        }
    }
    if (blockIdx.x == 0)
        reduce_edges<T, OP, false>(base + s.dst, base + s.src, s, pe_stride, npes, npes);
}

// Allreduce without LDS, for teams the LDS-staged kernel serves badly (more than 16 members: its block
// of 1024 threads leaves 32 or 16 lanes per member, i.e. 512 or 256 byte accesses): a block is ONE
// wavefront, lane i loads vector i of a 1 KiB piece from every member, eight loads in flight at a time,
// folds in member order and stores the result to every member.
// NPES > 0 fixes the team size at compile time (loads, fold and stores fully unrolled).
// ASTRIDE: streamed loads that share the lines at a tile's ends (as in the LDS-staged kernel's fetch).
template <typename T, int OP, int NPES, bool NTL, bool ASTRIDE = false>
__global__ __launch_bounds__(64) void reduce_gather_kernel(char *base, uint64_t slice_bytes,
                                                           const nvshmemi_amd_team_view_t *groups,
                                                           reduce_shape_t s) {
    constexpr int VEC = 16 / sizeof(T);
    constexpr int kBatch = 8;
    constexpr int kBatches = NPES ? (NPES + kBatch - 1) / kBatch : 1, kStores = NPES ? NPES : 1;  // unroll counts
    union pack_t {
        nvshmemi_v4u v;
        T e[VEC];
    };
    const nvshmemi_amd_team_view_t g = groups[blockIdx.z];
    const int npes = NPES ? NPES : g.size;
    base += (uint64_t)g.start * slice_bytes;
    const uint64_t pe_stride = (uint64_t)g.stride * slice_bytes;
    const uint64_t v = (uint64_t)dealt_tile(blockIdx.x, s.dealt) * 64 + threadIdx.x - s.lead;
    if (v < s.nvec) {
        const char *src = base + s.src + s.head * sizeof(T) + 16 * v;
        pack_t acc;
#pragma unroll kBatches
        for (int p0 = 0; p0 < npes; p0 += kBatch) {
            pack_t x[kBatch];
#pragma unroll
            for (int k = 0; k < kBatch; ++k)
                if (p0 + k < npes) {
                    const char *const from = src + (uint64_t)(p0 + k) * pe_stride;
                    x[k].v = ASTRIDE ? stream_load_astride(from, threadIdx.x - 8 >= 48) : stream_load<NTL>(from);
                }
#pragma unroll
            for (int k = 0; k < kBatch; ++k)
                if (p0 + k < npes) {
                    if (p0 + k == 0) {
                        acc = x[0];
                    } else {
#pragma unroll
                        for (int j = 0; j < VEC; ++j)
                            acc.e[j] = nvshmemi_amd_fold_step<T, OP>(p0 + k, acc.e[j], x[k].e[j]);
                    }
                }
        }
        char *dst = base + s.dst + s.head * sizeof(T) + 16 * v;
#pragma unroll kStores
        for (int p = 0; p < npes; ++p) stream_store<NVSHMEM_AMD_STORE_REDUCE>(dst + (uint64_t)p * pe_stride, acc.v);
    }
    if (blockIdx.x == 0)
        reduce_edges<T, OP, false>(base + s.dst, base + s.src, s, pe_stride, npes, npes);
}

// One element per lane and load, for small messages whose buffers are no whole vectors (element_at_a_time): what
// counts there is how long one lane is at work, and a lane of the vector kernels folds 2 to 16 elements, one after the
// other in 1- and 2-byte types, with the edges before or behind them.
template <typename T, int OP, bool SCATTER = false>
__global__ __launch_bounds__(256) void reduce_element_kernel(char *base, uint64_t slice_bytes,
                                                             const nvshmemi_amd_team_view_t *groups, uint64_t dst_off,
                                                             uint64_t src_off, uint64_t nelems) {
    const nvshmemi_amd_team_view_t g = groups[blockIdx.z];
    const int npes = g.size;
    if (SCATTER && (int)blockIdx.y >= npes) return;
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nelems) return;
    base += (uint64_t)g.start * slice_bytes;
    const uint64_t es = ((uint64_t)g.stride * slice_bytes) / sizeof(T);
    const T *s = reinterpret_cast<const T *>(base + src_off) + (SCATTER ? (uint64_t)blockIdx.y * nelems : 0);
    T *d = reinterpret_cast<T *>(base + dst_off) + (SCATTER ? (uint64_t)blockIdx.y * es : 0);
    T acc = s[i];
    for (int pe = 1; pe < npes; ++pe) acc = fold_next<T, OP, SCATTER>(pe, acc, s[(uint64_t)pe * es + i]);
    if (SCATTER) d[i] = acc;
    else for (int pe = 0; pe < npes; ++pe) d[(uint64_t)pe * es + i] = acc;
}

// reducescatter without LDS: a block is ONE wavefront, lane i loads vector i of a 1 KiB piece of block q
// (blockIdx.y) from every member - eight independent loads in flight per lane at a time - folds them in
// member order in registers and stores one vector into member q's destination.  The work is nearly all
// loads, and for loads this shape beats the LDS-staged tile of the allreduce: 6.3 against 5.9 TB/s for
// 8 members with 256 MiB of source each, 5.9 against 3.7 TB/s for 16 members.  NPES > 0 fixes the team
// size at compile time; NPES == 0 reads it from the team (16 members of bf16, sources of 6 | 12 | 24 MB in all, us
// unknown / known: 5.0 / 3.5, 5.5 / 4.2, 9.5 / 8.1; sixteen loads in flight gain them nothing more).
//
// Pieces are cut on the SOURCE's boundaries: n loads and one store per vector, so where blocks of an odd number of
// elements leave source and destination on different offsets, it is the store that straddles the lines and is
// unaligned.  Cut on the destination's, every load was, and each piece touched one line more of every member, which
// streamed loads fetch twice: us cached / streamed loads, 8 members of bf16 on odd elements, 100 MB of sources in all
// 23.7 / 22.8 then and 23.0 / 19.8 now, 200 MB 43.7 / 42.1 and 42.9 / 36.3 (aligned blocks: 42.0 / 36.0).
struct scatter_args_t {
    char *base;
    uint64_t slice_bytes;
    team_arg_t team;
    uint64_t dst, src;     // byte offsets of the destination and of the first source block in a slice
    uint64_t nelems;       // reduced here, of every block
    uint64_t block_bytes;  // from one source block to the next
};
// SCATTER false: the allreduce's operand order.
template <typename T, int OP, int NPES, bool NTL, bool SCATTER>
__device__ __forceinline__ void fold_source_pieces(const scatter_args_t &a) {
    constexpr int VEC = 16 / sizeof(T);
    constexpr int kBatch = 8;  // loads in flight per lane
    union pack_t {
        nvshmemi_v4u v;
        T e[VEC];
    };
    const nvshmemi_amd_team_view_t g = team_of(a.team, blockIdx.z);
    const int npes = NPES ? NPES : g.size;
    if ((int)blockIdx.y >= npes) return;
    char *const base = a.base + (uint64_t)g.start * a.slice_bytes;
    const uint64_t pe_stride = (uint64_t)g.stride * a.slice_bytes;
    const char *const block = base + a.src + (uint64_t)blockIdx.y * a.block_bytes;
    char *const dst = base + (uint64_t)blockIdx.y * pe_stride + a.dst;
    // whole vectors from the source's first 16-byte boundary on, and the elements around them
    uint64_t head = (-(uintptr_t)block & 15) / sizeof(T);
    if (head > a.nelems) head = a.nelems;
    const uint64_t nvec = (a.nelems - head) / VEC;
    if (blockIdx.x == 0) {
        const reduce_shape_t s = {0, 0, nvec, (uint32_t)head, (uint32_t)(a.nelems - head - nvec * VEC), 0, 0, false};
        reduce_edges<T, OP, SCATTER>(dst, block, s, pe_stride, npes, 1);
    }
    // pieces are cut on absolute 1 KiB boundaries: `lead` slots of piece 0 lie in front
    const char *const body = block + head * sizeof(T);
    const uint64_t lead = ((uint64_t)(uintptr_t)body >> 4) & 63;
    const uint64_t v = (uint64_t)blockIdx.x * 64 + threadIdx.x - lead;
    if (v >= nvec) return;  // also the slots in front of the block (wrapped)
    const char *src = body + 16 * v;
    pack_t acc;
    for (int p0 = 0; p0 < npes; p0 += kBatch) {
        pack_t x[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; ++k)
            if (p0 + k < npes) x[k].v = stream_load<NTL>(src + (uint64_t)(p0 + k) * pe_stride);
#pragma unroll
        for (int k = 0; k < kBatch; ++k)
            if (p0 + k < npes) {
                if (p0 + k == 0) {
                    acc = x[0];
                } else {
#pragma unroll
                    for (int j = 0; j < VEC; ++j) acc.e[j] = fold_next<T, OP, SCATTER>(p0 + k, acc.e[j], x[k].e[j]);
                }
            }
    }
    stream_store<NVSHMEM_AMD_STORE_REDUCESCATTER>(dst + head * sizeof(T) + 16 * v, acc.v);
}

template <typename T, int OP, int NPES, bool NTL>
__global__ __launch_bounds__(64) void reducescatter_gather_kernel(scatter_args_t a) {
    fold_source_pieces<T, OP, NPES, NTL, true>(a);
}
// The first half of the two-step allreduce of large teams: one block, into member 0's destination.  Always streamed: by
// default the form starts where streaming does (at exactly that size a byte earlier).
template <typename T, int OP>
__global__ __launch_bounds__(64) void reduce_root_kernel(scatter_args_t a) {
    fold_source_pieces<T, OP, 0, true, false>(a);
}

// Tiles of a segment, wherever it starts.
static uint64_t segment_tiles(uint64_t seg_bytes) { return (seg_bytes / 16 + 63 + 63) / 64; }

// members of all teams of the handle together
static uint64_t total_members(const TeamLaunch &tl) {
    // sizes lie between min and max; the exact sum only matters for the cache policy threshold
    return (uint64_t)tl.ngroups * (uint64_t)tl.max_size;
}

// How fcollect and broadcast store: paced beyond Runtime::paced_copy_blocks (33 to a compute unit: the 32 wavefronts it
// holds and what a message that is no power of two adds), up to which a grid is in flight all at once; from 12
// destinations on, whose stores are that many more, beyond half of that.  us paced / back to back at 1024, 4096, 6144,
// 8192 and 16384 blocks, buffers 5 bytes short of a power of two: fcollect to 4 members 3.4 / 2.7, 4.9 / 4.2, 6.1 / 5.4, 7.0
// / 6.4 and 11.9 / 11.6; to 8 4.7 / 3.4, 8.1 / 6.7, 10.4 / 9.2, 12.8 / 11.9 and 21.9 / 22.7; to 16 7.1 / 4.6, 14.8 / 12.4,
// 17.4 / 18.5, 24.0 / 24.2 and 43 / 47; broadcast to 8 4.2 / 3.0, 7.6 / 6.4, 9.6 / 9.2, 11.8 / 11.8 and 20.9 / 23.2, to 16 6.3
// / 4.2, 14.0 / 12.4, 17.8 / 18.8 and 22.5 / 24.4.  The times of 4096 blocks depend on where the buffers lie: with all of
// them at multiples of 16 MiB paced takes 6.6 to 8 and 11.2 to 16, back to back 6.5 and 12.0; everywhere else as above.
static bool paced_copy(const Runtime &rt, uint64_t blocks, int members) {
    return blocks > (members < 12 ? rt.paced_copy_blocks : rt.paced_copy_blocks / 2);
}
// Dynamic LDS that nobody uses: it limits the wavefronts of a paced copy that a compute unit (160 KiB) holds, and with
// them the width of each write front.  16 of the 32 possible while the cache holds the sources.  Streamed loads take
// longer and more wavefronts are needed to cover that: 24, and 28 from 12 destinations on, which keep a wavefront storing
// for longer.  us with 16 / 20 / 24 / 28 wavefronts, random data, sources | destinations in all.  Cached: fcollect 4 members
// 256 MiB | 1 GiB 178 / 183 / 186 / -, 8 members 128 MiB | 1 GiB 161 / 165 / 167 / -, 256 MiB | 2 GiB 322 / 328 / 332 / 334, 16
// members 128 MiB | 2 GiB 304 / 312 / 318 / 322; broadcast to 8 of 256 MiB 322 / 328 / 331 / -, to 16 of 64 MiB 156 / 155 / 160 /
// -.  Streamed: fcollect 8 members 512 MiB | 4 GiB 780 / 760 / 724 / 787, 12 members 384 MiB | 4.5 GiB 892 / 829 / 819 / 772, 16
// members 384 MiB | 6 GiB - / 1082 / 1044 / 1019, 512 MiB | 8 GiB - / 1446 / 1387 / 1429, 1 GiB | 16 GiB - / 2916 / 2794 / 2761,
// 32 members 512 MiB | 16 GiB - / 2681 / 2825 / 2610; broadcast of 512 MiB to 8 792 / 762 / 719 / 743, to 16 - / 1433 / 1359 /
// 1347.  (Medians; runs of one size spread by up to 8 % from 16 destinations on, with where the memory lies.)
static size_t paced_lds_bytes(const Runtime &rt, uint64_t source_bytes, int members) {
    const bool streamed = source_bytes > rt.cacheable_source_bytes;
    const unsigned waves = !streamed ? 16 : members < 12 ? 24 : 28;
    return ((size_t)160 << 10) / waves & ~(size_t)127;
}

// The blocks of an fcollect of streamed sources that walks in chunks, 0 for one that does not.  us chunked / paced: int64 of 16 x 32 MiB with all buffers at powers of two
// 1448 / 1526; elsewhere 16 x 32 MiB 1408 / 1429, 16 x 64 MiB 2782 / 2761, 24 x 16 MiB 1516 / 1552, 32 x 16 MiB 2745 / 2610 to
// 2930, with a third of the spread between runs; 12 x 32 MiB 816 / 772, 8 x 64 MiB 768 / 724.  Broadcasts and cached
// sources gain nothing by it (fcollect of 16 x 16 MiB 645 / 607).  The groups are the largest power of two that leaves each
// two destinations, the chunk 2^14 blocks over all groups, twice what the GPU holds at a time.
static uint64_t chunked_copy(segment_args_t *args, int members, uint64_t tiles) {
    if (members < 16) return 0;
    while (members >> (args->part_shift + 1) >= 2) ++args->part_shift;
    args->chunk_shift = (uint16_t)(14 - args->part_shift);
    const uint64_t chunks = (tiles + (1ull << args->chunk_shift) - 1) >> args->chunk_shift, blocks = chunks << 14;
    return blocks * 64 >> 32 ? 0 : blocks;  // (a launch holds fewer than 2^32 threads)
}

// Launches the broadcast kernel: member `root`'s [soff, +bytes) to every member's [doff, +bytes).
static int launch_broadcast(Runtime &rt, const TeamLaunch &tl, uint64_t doff, uint64_t soff, uint64_t bytes, int root,
                            hipStream_t stream) {
    const uint64_t tiles = segment_tiles(bytes), sources = bytes * (uint64_t)tl.ngroups;
    if (tiles > 0x7fffffffull) {
        set_error("broadcast: message too large");
        return NVSHMEMX_ERROR_INVALID_VALUE;
    }
    const dim3 grid((unsigned)tiles, 1, (unsigned)tl.ngroups);
    const segment_args_t args = {rt.base, rt.heap_size, team_arg(tl), doff, soff, bytes, (uint32_t)root,
                                 (uint32_t)tl.max_size, 0, 0, false};
    const bool paced = paced_copy(rt, tiles * (uint64_t)tl.ngroups, tl.max_size);
    const size_t lds = paced ? paced_lds_bytes(rt, sources, tl.max_size) : 0;
    // a source that cannot stay in the Infinity Cache is streamed
#define NVSHMEM_AMD_LAUNCH_BROADCAST(NTL, PACED)                                                                \
    launch_kernel((segment_copy_kernel<kModeBroadcast, NTL, PACED, NVSHMEM_AMD_STORE_REPLICATE>), grid,      \
                       dim3(64), lds, stream, args)
    if (!paced) NVSHMEM_AMD_LAUNCH_BROADCAST(false, false);
    else if (sources > rt.cacheable_source_bytes) NVSHMEM_AMD_LAUNCH_BROADCAST(true, true);
    else NVSHMEM_AMD_LAUNCH_BROADCAST(false, true);
#undef NVSHMEM_AMD_LAUNCH_BROADCAST
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("broadcast: kernel launch failed: %s", hipGetErrorString(e));
        return NVSHMEMX_ERROR_INTERNAL;
    }
    return 0;
}

// Whether a reduction that would take a gather kernel folds one element per lane instead.  Aligned buffers never do.
// Ragged ones with up to Runtime::element_reduce_bytes of results (512 KiB) do, except where the vector kernel is the
// faster one all the same: allreduces of 4- and 8-byte elements on 4 and more members, and teams whose size it knows at
// compile time, where it only loses 1- and 2-byte elements of up to 32 KiB (allreduce: 8 KiB) of results.
// us element / vector, allreduce of 4 KiB, 64 KiB, 512 KiB and 1 MiB: int8 on 2 members 2.0 / 3.3, 2.1 / 3.2, 3.2 / 3.4 and 4.8
// / 4.2, on 16 3.0 / 6.6, 3.3 / 6.3, 6.7 / 6.9 and 12.8 / 8.3, on 64 7.1 / 24, 8.1 / 23, 19 / 25 and 38 / 38; bf16 on 16 3.5 / 5.2,
// 3.6 / 5.0, 5.4 / 5.7 and 13.6 / 6.9; fp32 on 2 2.0 / 2.6, 2.1 / 2.4, 2.4 / 2.6 and 2.8 / 2.9, on 3 2.4 / 2.7, 2.4 / 2.7, 2.7 /
// 2.8, on 16 4.6 / 3.6, 4.7 / 3.6, 6.0 / 4.3; int8 on 8 2.5 / 2.6, 2.9 / 2.7.  reducescatter with 32 KiB and 512 KiB of results
// in all: int8 on 4 members 2.4 / 3.5 and 3.5 / 3.6, on 16 3.0 / 6.5 and 4.4 / 6.4, on 8 2.6 / 2.8 and 4.1 / 2.9; fp32 on 4
// 2.4 / 2.6 and 2.6 / 2.8, on 16 3.4 / 3.7 and 3.5 / 3.7.
template <typename T, bool SCATTER>
bool element_at_a_time(const Runtime &rt, const TeamLaunch &tl, bool known_size, uint64_t dst_off, uint64_t src_off,
                       uint64_t nelems) {
    const uint64_t bytes = nelems * sizeof(T), results = SCATTER ? bytes * (uint64_t)tl.max_size : bytes;
    if (((dst_off | src_off | (SCATTER ? bytes : 0)) & 15) == 0) return false;
    if (known_size) return sizeof(T) <= 2 && results <= rt.element_reduce_bytes / (SCATTER ? 16 : 64);
    return (SCATTER || sizeof(T) <= 2 || tl.max_size <= 3) && results <= rt.element_reduce_bytes;
}

template <typename T, int OP>
void launch_reduce(Runtime &rt, const TeamLaunch &tl, uint64_t dst_off, uint64_t src_off,
                   uint64_t nelems, uint64_t all, hipStream_t stream) {
    const unsigned ngroups = (unsigned)tl.ngroups;
    reduce_shape_t shape = reduce_shape<T>(rt, dst_off, src_off, nelems);
    const uint64_t nvec = shape.nvec;
    // Which kernel.  From Runtime::lds_reduce_bytes of sources in all (64 MiB; a quarter
    // of that for teams of 17 to 32 members, four times for larger ones) the LDS-staged
    // kernel wins for every team of 3 to 64 members; below that, and for 2 members, the gather kernel does.
    // fp32 sum on a stream, LDS-staged / gather in TB/s, sources of 32 MiB | 64 MiB | 128 MiB in all: 4 members
    // 7.3 / 8.4 | 7.6 / 7.4 | 8.3 / 8.1, 8 members 7.8 / 8.3 | 7.8 / 6.9 | 8.5 / 7.7, 16 members 7.0 / 8.3 |
    // 7.6 / 6.6 | 8.3 / 7.6; 32 members lead with the LDS kernel from 16 MiB on (7.3 / 5.3), 48 and 64 members
    // with the gather kernel up to 128-192 MiB (5.9 / 6.8).  Beyond the cache,
    // measured with random fp32 data and write-through stores, LDS-staged against gather, TB/s at
    // 512 MiB / 2 GiB of sources: 4 members 6.54 / 6.55 against 6.19 / 6.24, 6 members 6.37 / 6.44
    // against 5.89 / 5.58, 8 members 6.46 / 6.53 against 6.03 / 6.09, 12 members 6.28 / 6.28 against
    // 5.73 / 5.83, 16 members 6.21 / 6.12 against 5.44 / 5.57, 32 members 6.17 / 6.10 against 5.22 / 5.49,
    // 64 members 5.64 / 5.64 against 5.15 / 5.26.  A wavefront of the LDS kernel serves
    //   4 members   one                                        (team size known at compile time)
    //   8 members   one; cached sources of 1- and 2-byte elements two   (known)
    //   16 members  cached: one, 1- and 2-byte elements two    (known); streamed: two
    //   32 members  two                                        (cached: known)
    //   others      two up to 32 members, four beyond (there: handles whose smallest team has fewer than
    //               two_step_reduce_members, and programs without the two-step form)
    // One load and one store per lane measured best where the block stays within 16 wavefronts (narrow elements:
    // NVSHMEM_AMD_REDUCE_NARROW_MPW), and wavefronts of fewer than 64 lanes per member (512- or 256-byte accesses) lost
    // 7-22 % against the gather kernel.  The compile-time size is worth 6 % at 32 members (6.17 against 5.82), nothing at 64,
    // and with a member per wavefront 3 to 8 % at 4 (70 | 200 | 800 MB of sources in all, fp32 22.4 / 20.9 | 63.6 / 61.8 | 248 / 240
    // us, bf16 alike).  Streamed sources of 16 and 32 members take two steps (below); for programs that switch those off the size read
    // from the team does, us known / read, 110 | 200 | 600 MB in turn: 16 members fp32 38.5 / 39.0 | 67.4 / 68.0 | 193.6 / 198.0, bf16 39.7 /
    // 39.1 | 69.0 / 68.3 | 201.2 / 198.4, 32 members fp32 40.3 / 41.4 | 69.5 / 71.8 | 207.1 / 212.7.
    const uint64_t total_bytes = total_members(tl) * all * sizeof(T);
    const int fixed_size = tl.min_size == tl.max_size ? tl.max_size : 0;
    const bool stream_source = rt.streamed_reduction(total_bytes);
    // (in bytes whatever the element type: fp32, bf16 and int64 cross over at the same 64 MiB on 8 and 16 members)
    const uint64_t lds_from_bytes = tl.max_size > 32   ? rt.lds_reduce_bytes * 4
                                    : tl.max_size > 16 ? rt.lds_reduce_bytes / 4
                                                       : rt.lds_reduce_bytes;
    // mpw: members per wavefront of the LDS-staged kernel; ct_size: a compile-time team size, if any
    int mpw = 0, ct_size = 0;
    constexpr int kNarrowMpw = sizeof(T) <= 2 ? NVSHMEM_AMD_REDUCE_NARROW_MPW : NVSHMEM_AMD_REDUCE_WIDE_MPW;
    if (fixed_size == 8) ct_size = 8, mpw = stream_source ? NVSHMEM_AMD_REDUCE_WIDE_MPW : kNarrowMpw;
    else if (fixed_size == 4) ct_size = 4, mpw = 1;
    else if (fixed_size == 16 && !stream_source) ct_size = 16, mpw = kNarrowMpw;
    else if (fixed_size == 32 && !stream_source) ct_size = 32, mpw = 2;
    else if (tl.max_size >= 3 && tl.max_size <= 32) mpw = 2;
    else if (tl.max_size > 32 && tl.max_size <= 64) mpw = 4;
    // Two-step allreduce of large teams: fold into member 0's destination (n loads and ONE store per vector, the
    // shape of the reducescatter), then broadcast that.  It moves 2 n + 2 units where the fused
    // kernel moves 2 n, but every block of the fused kernel feeds n write fronts of 1 KiB pieces, and its fold
    // serialises n steps between two barriers.  fp32 sum of random data, TB/s, fused / two-step at about 512 MiB and 2 to
    // 4 GiB of sources in all: 12 members 6.02 / 6.03 and 6.23 / 6.20, 16: 6.12 / 6.25 and 6.12 / 6.32, 24: 5.72 / 6.24 and 5.79 /
    // 6.39, 32: 6.28 / 6.19 and 6.35 / 6.42, 48: 5.87 / 6.38 and 5.94 / 6.47, 64: 5.86 / 5.81 and 6.01 / 6.47; at 256 MiB 16
    // members 6.98 / 6.10, 32 6.93 / 6.27, 64 6.37 / 6.31 for a source that is reduced again as it is.  Other buffers in turn,
    // us fused / two-step, 104 | 160 | 240 MB of sources in all: 16 members fp32 51.6 / 37.1 | 75.8 / 55.4 | 95.3 / 78.7, bf16 50.0 / 38.3 |
    // 68.3 / 56.7 | 96.5 / 79.8, 24 fp32 40.4 / 40.6 | 59.6 / 53.7 | 88.6 / 80.6, 32 48.9 / 40.0 | 69.6 / 61.4 | 99.7 / 79.9, against the gather
    // kernel 40 39.5 / 38.4 | 63.0 / 58.8 | 93.1 / 81.4, 64 42.4 / 41.9 | 64.7 / 59.2 | 98.3 / 88.9; sources that are still in the cache lose
    // (16 members, 80 MB: 26.8 / 31.5).  So: from Runtime::two_step_reduce_members (16) members on when the sources hold
    // two_step_reduce_bytes or more (96 MiB, from where reductions stream; with a larger cacheable_source_bytes 3/8 of that).
    if (rt.two_step_reduce_members && tl.min_size >= (int)rt.two_step_reduce_members && total_bytes >= rt.two_step_reduce_bytes) {
        const scatter_args_t args = {rt.base, rt.heap_size, team_arg(tl), dst_off, src_off, nelems, 0};
        const dim3 grid((unsigned)((nelems / (16 / sizeof(T)) + 63 + 63) / 64), 1, ngroups);
        launch_kernel((reduce_root_kernel<T, OP>), grid, dim3(64), 0, stream, args);
        (void)launch_broadcast(rt, tl, dst_off, dst_off, nelems * sizeof(T), 0, stream);
        return;
    }
    if (mpw && total_bytes >= lds_from_bytes) {
        const uint32_t lane_shift = 6;
        const unsigned threads = (unsigned)((tl.max_size + mpw - 1) / mpw) << lane_shift;
        // A tile of two vectors per thread halves the barriers per byte and loses all the same: 4-byte and 8-byte elements 3-4 %;
        // bf16 on 8 members, streamed with a member per wavefront, one / two vectors, us at 110 | 200 | 400 | 1600 MB of sources in all
        // in turn 42.5 / 44.6 | 68.5 / 72.6 | 131.8 / 143.8 | 517 / 581.
        constexpr int kVptNarrow = sizeof(T) <= 2 ? NVSHMEM_AMD_REDUCE_VPT_NARROW : NVSHMEM_AMD_REDUCE_VPT;
        const int vpt = (ct_size == 8 || ct_size == 16) ? kVptNarrow : NVSHMEM_AMD_REDUCE_VPT;
        const uint64_t tile_vecs = (uint64_t)vpt << lane_shift;
        const uint64_t blocks = (nvec + (1u << lane_shift) + tile_vecs - 1) / tile_vecs;  // room for the lead-in
        shape.dealt = dealt_blocks(dst_off, src_off, blocks);
        shape.astride = (dst_off - src_off) % 128 && total_bytes <= rt.cacheable_source_bytes;
        const size_t lds = ((size_t)tl.max_size + 1) * 16 * tile_vecs;
        const dim3 grid((unsigned)blocks, 1, ngroups);
#define NVSHMEM_AMD_LAUNCH_REDUCE(N, NTL, MPW, VPT)                                                      \
    launch_kernel((reduce_vector_kernel<T, OP, N, NTL, VPT, MPW>), grid, dim3(threads), lds, stream, rt.base, \
                  rt.heap_size, tl.groups, shape)
#define NVSHMEM_AMD_LAUNCH_REDUCE_EITHER(N, MPW)                                          \
    do {                                                                                  \
        if (stream_source) NVSHMEM_AMD_LAUNCH_REDUCE(N, true, MPW, NVSHMEM_AMD_REDUCE_VPT); \
        else NVSHMEM_AMD_LAUNCH_REDUCE(N, false, MPW, NVSHMEM_AMD_REDUCE_VPT);              \
    } while (0)
        if (ct_size == 8 && stream_source) NVSHMEM_AMD_LAUNCH_REDUCE(8, true, NVSHMEM_AMD_REDUCE_WIDE_MPW, kVptNarrow);
        else if (ct_size == 8) NVSHMEM_AMD_LAUNCH_REDUCE(8, false, kNarrowMpw, kVptNarrow);
        else if (ct_size == 16) NVSHMEM_AMD_LAUNCH_REDUCE(16, false, kNarrowMpw, kVptNarrow);
        else if (ct_size == 32) NVSHMEM_AMD_LAUNCH_REDUCE(32, false, 2, NVSHMEM_AMD_REDUCE_VPT);
        else if (ct_size == 4) NVSHMEM_AMD_LAUNCH_REDUCE_EITHER(4, 1);
        else if (mpw == 2) NVSHMEM_AMD_LAUNCH_REDUCE_EITHER(0, 2);
        else NVSHMEM_AMD_LAUNCH_REDUCE_EITHER(0, 4);
#undef NVSHMEM_AMD_LAUNCH_REDUCE_EITHER
#undef NVSHMEM_AMD_LAUNCH_REDUCE
    } else if (element_at_a_time<T, false>(rt, tl, fixed_size == 4 || fixed_size == 8, dst_off, src_off, nelems)) {
        launch_kernel((reduce_element_kernel<T, OP>), dim3((unsigned)((nelems + 255) / 256), 1, ngroups), dim3(256), 0,
                           stream, rt.base, rt.heap_size, tl.groups, dst_off, src_off, nelems);
    } else {
        // room for the lead-in; at least one block for the edges
        const dim3 grid((unsigned)((nvec + 63 + 63) / 64), 1, ngroups);
        shape.dealt = dealt_blocks(dst_off, src_off, grid.x);
        const bool astride = stream_source && (dst_off - src_off) % 128 && total_bytes <= rt.cacheable_source_bytes;
#define NVSHMEM_AMD_LAUNCH_GATHER_REDUCE(...)                                                                          \
    launch_kernel((reduce_gather_kernel<T, OP, __VA_ARGS__>), grid, dim3(64), 0, stream, rt.base, rt.heap_size, tl.groups, shape)
        // (streamed sources of 4 and 8 members come here only with a larger NVSHMEM_AMD_LDS_REDUCE_BYTES; sixteen members
        // unrolled measured slower than the loop: 5.2 against 5.4 TB/s)
        if (astride) NVSHMEM_AMD_LAUNCH_GATHER_REDUCE(0, true, true);
        else if (stream_source) NVSHMEM_AMD_LAUNCH_GATHER_REDUCE(0, true);
        else if (fixed_size == 4) NVSHMEM_AMD_LAUNCH_GATHER_REDUCE(4, false);
        else if (fixed_size == 8) NVSHMEM_AMD_LAUNCH_GATHER_REDUCE(8, false);
        else NVSHMEM_AMD_LAUNCH_GATHER_REDUCE(0, false);
#undef NVSHMEM_AMD_LAUNCH_GATHER_REDUCE
    }
}

// reducescatter: grid.y = destination member; nelems of the `all` elements of one PE's result
template <typename T, int OP>
void launch_reducescatter(Runtime &rt, const TeamLaunch &tl, uint64_t dst_off, uint64_t src_off,
                          uint64_t nelems, uint64_t all, hipStream_t stream) {
    const bool eight = tl.min_size == 8 && tl.max_size == 8;
    if (nelems == all && element_at_a_time<T, true>(rt, tl, eight, dst_off, src_off, nelems)) {
        const dim3 grid((unsigned)((nelems + 255) / 256), (unsigned)tl.max_size, (unsigned)tl.ngroups);
        launch_kernel((reduce_element_kernel<T, OP, true>), grid, dim3(256), 0, stream, rt.base, rt.heap_size,
                           tl.groups, dst_off, src_off, nelems);
        return;
    }
    const scatter_args_t args = {rt.base, rt.heap_size, team_arg(tl), dst_off, src_off, nelems, all * sizeof(T)};
    const uint64_t blocks = (nelems / (16 / sizeof(T)) + 63 + 63) / 64;  // room for the lead-in; at least one block for the edges
    const dim3 grid((unsigned)blocks, (unsigned)tl.max_size, (unsigned)tl.ngroups);
    const bool stream_source = rt.streamed_reduction(total_members(tl) * tl.max_size * all * sizeof(T));
#define NVSHMEM_AMD_LAUNCH_GATHER(N)                                                                                   \
    do {                                                                                                               \
        if (stream_source)                                                                                             \
            launch_kernel((reducescatter_gather_kernel<T, OP, N, true>), grid, dim3(64), 0, stream, args);        \
        else                                                                                                           \
            launch_kernel((reducescatter_gather_kernel<T, OP, N, false>), grid, dim3(64), 0, stream, args);       \
    } while (0)
    if (eight) NVSHMEM_AMD_LAUNCH_GATHER(8);
    else if (tl.min_size == 16 && tl.max_size == 16) NVSHMEM_AMD_LAUNCH_GATHER(16);
    else NVSHMEM_AMD_LAUNCH_GATHER(0);
#undef NVSHMEM_AMD_LAUNCH_GATHER
}

typedef void (*reduce_launcher_t)(Runtime &, const TeamLaunch &, uint64_t, uint64_t, uint64_t, uint64_t, hipStream_t);

// A launch holds fewer than 2^32 threads, and the LDS-staged kernel has up to 1024 of them for every KiB of one PE's
// result: a reduction goes out in pieces of 2 GiB per PE, of 2^21 blocks.
constexpr uint64_t kReducePieceBytes = (uint64_t)2 << 30;
void launch_pieces(reduce_launcher_t fn, Runtime &rt, const TeamLaunch &tl, uint64_t doff, uint64_t soff, uint64_t nelems,
                   size_t es, hipStream_t stream) {
    const uint64_t piece = kReducePieceBytes / es;
    for (uint64_t done = 0; done < nelems; done += piece)
        fn(rt, tl, doff + done * es, soff + done * es, nelems - done < piece ? nelems - done : piece, nelems, stream);
}

template <typename T, bool SCATTER>
reduce_launcher_t pick_arith(int op) {
#define NVSHMEM_AMD_PICK(OP) \
    case NVSHMEMI_OP_##OP: return SCATTER ? launch_reducescatter<T, NVSHMEMI_OP_##OP> : launch_reduce<T, NVSHMEMI_OP_##OP>
    switch (op) {
        NVSHMEM_AMD_PICK(min);
        NVSHMEM_AMD_PICK(max);
        NVSHMEM_AMD_PICK(sum);
        NVSHMEM_AMD_PICK(prod);
        default: return nullptr;
    }
}
template <typename T, bool SCATTER>
reduce_launcher_t pick_integer(int op) {
    switch (op) {
        NVSHMEM_AMD_PICK(and);
        NVSHMEM_AMD_PICK(or);
        NVSHMEM_AMD_PICK(xor);
        default: return pick_arith<T, SCATTER>(op);
    }
#undef NVSHMEM_AMD_PICK
}

template <bool SCATTER>
reduce_launcher_t pick_reduce(int dtype, int op) {
    switch (dtype) {
        case NVSHMEMI_DT_i8: return pick_integer<int8_t, SCATTER>(op);
        case NVSHMEMI_DT_i16: return pick_integer<int16_t, SCATTER>(op);
        case NVSHMEMI_DT_i32: return pick_integer<int32_t, SCATTER>(op);
        case NVSHMEMI_DT_i64: return pick_integer<int64_t, SCATTER>(op);
        case NVSHMEMI_DT_u8: return pick_integer<uint8_t, SCATTER>(op);
        case NVSHMEMI_DT_u16: return pick_integer<uint16_t, SCATTER>(op);
        case NVSHMEMI_DT_u32: return pick_integer<uint32_t, SCATTER>(op);
        case NVSHMEMI_DT_u64: return pick_integer<uint64_t, SCATTER>(op);
        case NVSHMEMI_DT_f16: return pick_arith<__half, SCATTER>(op);
        case NVSHMEMI_DT_bf16: return pick_arith<__hip_bfloat16, SCATTER>(op);
        case NVSHMEMI_DT_f32: return pick_arith<float, SCATTER>(op);
        case NVSHMEMI_DT_f64: return pick_arith<double, SCATTER>(op);
        default: return nullptr;
    }
}

const size_t kDtypeSize[NVSHMEMI_DT_COUNT] = {1, 2, 4, 8, 1, 2, 4, 8, 2, 2, 4, 8};

}  // namespace

int reduce_on_stream(int dtype, int op, nvshmem_team_t team, void *dest, const void *src,
                     size_t nreduce, hipStream_t stream) {
    Runtime &rt = Runtime::get();
    std::lock_guard<std::recursive_mutex> lock(rt.mu);
    TeamLaunch tl;
    if (!resolve_team(rt, "reduce", team, &tl)) return NVSHMEMX_ERROR_INVALID_VALUE;
    reduce_launcher_t fn = pick_reduce<false>(dtype, op);
    if (!fn) {
        set_error("reduce: operator %d is not defined for element kind %d", op, dtype);
        return NVSHMEMX_ERROR_INVALID_VALUE;
    }
    if (nreduce == 0) return 0;
    const size_t es = kDtypeSize[dtype];
    uint64_t doff = 0, soff = 0;
    if (nreduce > rt.heap_size / es) {
        set_error("reduce: %zu elements of %zu bytes leave the PE's heap slice", nreduce, es);
        return NVSHMEMX_ERROR_INVALID_VALUE;
    }
    if (!check_symmetric_range(rt, "reduce dest", dest, nreduce * es, &doff) ||
        !check_symmetric_range(rt, "reduce source", src, nreduce * es, &soff))
        return NVSHMEMX_ERROR_INVALID_VALUE;
    if ((doff % es) || (soff % es)) {
        set_error("reduce: buffers must be aligned to the element size");
        return NVSHMEMX_ERROR_INVALID_VALUE;
    }
    if (doff != soff && doff < soff + nreduce * es && soff < doff + nreduce * es) {
        set_error("reduce: dest and source overlap without being identical");
        return NVSHMEMX_ERROR_INVALID_VALUE;
    }
    launch_pieces(fn, rt, tl, doff, soff, nreduce, es, stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("reduce: kernel launch failed: %s", hipGetErrorString(e));
        return NVSHMEMX_ERROR_INTERNAL;
    }
    return 0;
}

int reducescatter_on_stream(int dtype, int op, nvshmem_team_t team, void *dest, const void *src,
                            size_t nreduce, hipStream_t stream) {
    Runtime &rt = Runtime::get();
    std::lock_guard<std::recursive_mutex> lock(rt.mu);
    TeamLaunch tl;
    if (!resolve_team(rt, "reducescatter", team, &tl)) return NVSHMEMX_ERROR_INVALID_VALUE;
    reduce_launcher_t fn = pick_reduce<true>(dtype, op);
    if (!fn) {
        set_error("reducescatter: operator %d is not defined for element kind %d", op, dtype);
        return NVSHMEMX_ERROR_INVALID_VALUE;
    }
    if (nreduce == 0) return 0;
    const size_t es = kDtypeSize[dtype];
    const uint64_t n = (uint64_t)tl.max_size;
    if (nreduce > rt.heap_size / es / n) {
        set_error("reducescatter: %zu elements of %zu bytes x %d PEs leave the PE's heap slice",
                  nreduce, es, tl.max_size);
        return NVSHMEMX_ERROR_INVALID_VALUE;
    }
    uint64_t doff = 0, soff = 0;
    if (!check_symmetric_range(rt, "reducescatter dest", dest, nreduce * es, &doff) ||
        !check_symmetric_range(rt, "reducescatter source", src, nreduce * es * n, &soff))
        return NVSHMEMX_ERROR_INVALID_VALUE;
    if ((doff % es) || (soff % es)) {
        set_error("reducescatter: buffers must be aligned to the element size");
        return NVSHMEMX_ERROR_INVALID_VALUE;
    }
    // PE q writes dest while other PEs' blocks of the source at the same offsets are still read
    if (doff < soff + nreduce * es * n && soff < doff + nreduce * es) {
        set_error("reducescatter: dest and source overlap");
        return NVSHMEMX_ERROR_INVALID_VALUE;
    }
    launch_pieces(fn, rt, tl, doff, soff, nreduce, es, stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("reducescatter: kernel launch failed: %s", hipGetErrorString(e));
        return NVSHMEMX_ERROR_INTERNAL;
    }
    return 0;
}

int broadcast_on_stream(nvshmem_team_t team, void *dest, const void *src, size_t bytes, int root,
                        hipStream_t stream) {
    Runtime &rt = Runtime::get();
    std::lock_guard<std::recursive_mutex> lock(rt.mu);
    TeamLaunch tl;
    if (!resolve_team(rt, "broadcast", team, &tl)) return NVSHMEMX_ERROR_INVALID_VALUE;
    if (root < 0 || root >= tl.min_size) {
        set_error("broadcast: root %d is not a PE of the team (0..%d)", root, tl.min_size - 1);
        return NVSHMEMX_ERROR_INVALID_VALUE;
    }
    if (bytes == 0) return 0;
    uint64_t doff = 0, soff = 0;
    if (!check_symmetric_range(rt, "broadcast dest", dest, bytes, &doff) ||
        !check_symmetric_range(rt, "broadcast source", src, bytes, &soff))
        return NVSHMEMX_ERROR_INVALID_VALUE;
    // identical buffers are the in-place form (the root keeps its data); a partial overlap would
    // let the root's destination clobber source bytes that are still to be read
    if (doff != soff && doff < soff + bytes && soff < doff + bytes) {
        set_error("broadcast: dest and source overlap without being identical");
        return NVSHMEMX_ERROR_INVALID_VALUE;
    }
    return launch_broadcast(rt, tl, doff, soff, bytes, root, stream);
}

static int segment_collective(int mode, const char *what, nvshmem_team_t team, void *dest,
                              const void *src, size_t seg_bytes, hipStream_t stream) {
    Runtime &rt = Runtime::get();
    std::lock_guard<std::recursive_mutex> lock(rt.mu);
    TeamLaunch tl;
    if (!resolve_team(rt, what, team, &tl)) return NVSHMEMX_ERROR_INVALID_VALUE;
    if (seg_bytes == 0) return 0;
    const uint64_t n = (uint64_t)tl.max_size;
    if (seg_bytes > rt.heap_size / n) {
        set_error("%s: %zu bytes x %d PEs does not fit a PE's heap slice", what, seg_bytes, tl.max_size);
        return NVSHMEMX_ERROR_INVALID_VALUE;
    }
    const uint64_t src_bytes = mode == kModeFcollect ? seg_bytes : seg_bytes * n;
    uint64_t doff = 0, soff = 0;
    if (!check_symmetric_range(rt, what, dest, seg_bytes * n, &doff) ||
        !check_symmetric_range(rt, what, src, src_bytes, &soff))
        return NVSHMEMX_ERROR_INVALID_VALUE;
    if (doff < soff + src_bytes && soff < doff + seg_bytes * n) {
        set_error("%s: dest and source overlap", what);
        return NVSHMEMX_ERROR_INVALID_VALUE;
    }
    const uint64_t tiles = segment_tiles(seg_bytes), sources = src_bytes * total_members(tl);
    if (tiles > 0x7fffffffull) {
        set_error("%s: message too large", what);
        return NVSHMEMX_ERROR_INVALID_VALUE;
    }
    // Alltoalls of 7/16 (112 MiB) to all of what the Infinity Cache could hold stream three quarters of a source and keep a
    // quarter, the lines at the ends of its pieces, which on another offset than the destination's two wavefronts read.  Beside
    // other buffers in turn a source kept whole is gone when it comes again, a quarter is not.  us kept / a quarter kept, fp32
    // normal data, 120 | 200 | 240 | 256 MiB of sources in all, 8 members, three sets of buffers in turn 39.2 / 36.5 | 66.3 / 59.3 | 79.5 /
    // 70.5 | 84.5 / 75.2, each filled in front of its call (both kernels) 74.5 / 70.6 | 110.0 / 107.0 | 124.8 / 125.8 | 129.0 / 133.4; what
    // loses is a source sent again as it is, with nothing in between: 34.9 / 36.2 | 58.2 / 59.6 | 68.6 / 70.2 | 72.8 / 75.3.  256 MiB on 4
    // and 16 members: in turn 84.4 / 74.8 and 84.5 / 77.5, filled 117.9 / 118.8 and 143.1 / 146.8, again as it is 72.8 / 74.7 and 72.4 /
    // 77.8; on another offset, 8 members, 85.2 / 80.7, 132.5 / 136.2 and 76.0 / 80.6.  None kept: 200 MiB in turn 63.3.  Below 112
    // MiB three buffers in turn are still there in part: 105 MB 31.9 / 31.2, on another offset 33.2 / 33.4, 16 members 37.2 / 38.8.
    // (Dealing the tiles to the XCDs, as in the reductions, loses 2 % here.)
    const bool quarter = mode == kModeAlltoall && sources > rt.cacheable_source_bytes / 16 * 7 && sources <= rt.cacheable_source_bytes;
    const bool stream_source = quarter || sources > rt.cacheable_source_bytes;
    const segment_args_t args = {rt.base, rt.heap_size, team_arg(tl), doff, soff, seg_bytes, 0, (uint32_t)n, 0, 0, quarter};
#define NVSHMEM_AMD_LAUNCH_SEGCOPY(MODE, NTL, PACED, STORE) \
    launch_kernel((segment_copy_kernel<MODE, NTL, PACED, STORE>), grid, dim3(64), lds, stream, args)
    if (mode == kModeFcollect) {
        const dim3 grid((unsigned)tiles, (unsigned)n, (unsigned)tl.ngroups);
        const bool paced = paced_copy(rt, tiles * n * (uint64_t)tl.ngroups, tl.max_size);
        const size_t lds = paced ? paced_lds_bytes(rt, sources, tl.max_size) : 0;
        segment_args_t chunked = args;
        const uint64_t chunked_blocks = paced && stream_source ? chunked_copy(&chunked, tl.max_size, tiles) : 0;
        if (chunked_blocks) {
            launch_kernel((segment_copy_kernel<kModeFcollect, false, true, NVSHMEM_AMD_STORE_REPLICATE, true>),
                               dim3((unsigned)chunked_blocks, grid.y, grid.z), dim3(64), 0, stream, chunked);
        } else if (!paced) NVSHMEM_AMD_LAUNCH_SEGCOPY(kModeFcollect, false, false, NVSHMEM_AMD_STORE_REPLICATE);
        else if (stream_source) NVSHMEM_AMD_LAUNCH_SEGCOPY(kModeFcollect, true, true, NVSHMEM_AMD_STORE_REPLICATE);
        else NVSHMEM_AMD_LAUNCH_SEGCOPY(kModeFcollect, false, true, NVSHMEM_AMD_STORE_REPLICATE);
    } else {
        const dim3 grid((unsigned)tiles, (unsigned)n, (unsigned)(n * tl.ngroups));
        const size_t lds = 0;  // (one store per load: every wavefront counts)
        if (stream_source) NVSHMEM_AMD_LAUNCH_SEGCOPY(kModeAlltoall, true, false, NVSHMEM_AMD_STORE_ALLTOALL);
        else NVSHMEM_AMD_LAUNCH_SEGCOPY(kModeAlltoall, false, false, NVSHMEM_AMD_STORE_ALLTOALL);
    }
#undef NVSHMEM_AMD_LAUNCH_SEGCOPY
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("%s: kernel launch failed: %s", what, hipGetErrorString(e));
        return NVSHMEMX_ERROR_INTERNAL;
    }
    return 0;
}

int fcollect_on_stream(nvshmem_team_t team, void *dest, const void *src, size_t bytes,
                       hipStream_t stream) {
    return segment_collective(kModeFcollect, "fcollect", team, dest, src, bytes, stream);
}
int alltoall_on_stream(nvshmem_team_t team, void *dest, const void *src, size_t bytes,
                       hipStream_t stream) {
    return segment_collective(kModeAlltoall, "alltoall", team, dest, src, bytes, stream);
}

static int finish_blocking(int rc) {
    if (rc == 0) NVSHMEM_AMD_HIP_CHECK(hipStreamSynchronize(nullptr));
    return rc;
}

}  // namespace nvshmem_amd

using namespace nvshmem_amd;

extern "C" {

#define NVSHMEMI_DEFINE_TYPED_COLL_HOST(NAME, TYPE, TAG)                                          \
    int nvshmemx_##NAME##_alltoall_on_stream(nvshmem_team_t team, TYPE *dest, const TYPE *src,    \
                                             size_t nelems, nvshmemx_stream_t s) {                \
        return alltoall_on_stream(team, dest, src, nelems * sizeof(TYPE), (hipStream_t)s);        \
    }                                                                                             \
    int nvshmemx_##NAME##_fcollect_on_stream(nvshmem_team_t team, TYPE *dest, const TYPE *src,    \
                                             size_t nelems, nvshmemx_stream_t s) {                \
        return fcollect_on_stream(team, dest, src, nelems * sizeof(TYPE), (hipStream_t)s);        \
    }                                                                                             \
    int nvshmemx_##NAME##_broadcast_on_stream(nvshmem_team_t team, TYPE *dest, const TYPE *src,   \
                                              size_t nelems, int PE_root, nvshmemx_stream_t s) {  \
        return broadcast_on_stream(team, dest, src, nelems * sizeof(TYPE), PE_root,               \
                                   (hipStream_t)s);                                               \
    }                                                                                             \
    int nvshmem_##NAME##_broadcast(nvshmem_team_t team, TYPE *dest, const TYPE *src,              \
                                   size_t nelems, int PE_root) {                                  \
        return finish_blocking(                                                                   \
            broadcast_on_stream(team, dest, src, nelems * sizeof(TYPE), PE_root, nullptr));       \
    }                                                                                             \
    int nvshmem_##NAME##_alltoall(nvshmem_team_t team, TYPE *dest, const TYPE *src,               \
                                  size_t nelems) {                                                \
        return finish_blocking(                                                                   \
            alltoall_on_stream(team, dest, src, nelems * sizeof(TYPE), nullptr));                 \
    }                                                                                             \
    int nvshmem_##NAME##_fcollect(nvshmem_team_t team, TYPE *dest, const TYPE *src,               \
                                  size_t nelems) {                                                \
        return finish_blocking(                                                                   \
            fcollect_on_stream(team, dest, src, nelems * sizeof(TYPE), nullptr));                 \
    }
NVSHMEMI_REPT_FOR_STANDARD_RMA_TYPES(NVSHMEMI_DEFINE_TYPED_COLL_HOST)
#undef NVSHMEMI_DEFINE_TYPED_COLL_HOST

int nvshmemx_alltoallmem_on_stream(nvshmem_team_t team, void *dest, const void *src, size_t nelems,
                                   nvshmemx_stream_t stream) {
    return alltoall_on_stream(team, dest, src, nelems, (hipStream_t)stream);
}
int nvshmemx_fcollectmem_on_stream(nvshmem_team_t team, void *dest, const void *src, size_t nelems,
                                   nvshmemx_stream_t stream) {
    return fcollect_on_stream(team, dest, src, nelems, (hipStream_t)stream);
}
int nvshmemx_broadcastmem_on_stream(nvshmem_team_t team, void *dest, const void *src, size_t nelems,
                                    int PE_root, nvshmemx_stream_t stream) {
    return broadcast_on_stream(team, dest, src, nelems, PE_root, (hipStream_t)stream);
}
int nvshmem_broadcastmem(nvshmem_team_t team, void *dest, const void *src, size_t nelems,
                         int PE_root) {
    return finish_blocking(broadcast_on_stream(team, dest, src, nelems, PE_root, nullptr));
}
int nvshmem_alltoallmem(nvshmem_team_t team, void *dest, const void *src, size_t nelems) {
    return finish_blocking(alltoall_on_stream(team, dest, src, nelems, nullptr));
}
int nvshmem_fcollectmem(nvshmem_team_t team, void *dest, const void *src, size_t nelems) {
    return finish_blocking(fcollect_on_stream(team, dest, src, nelems, nullptr));
}

#define NVSHMEMI_DEFINE_TYPED_REDUCE_HOST(NAME, TYPE, TAG, OP)                                    \
    int nvshmemx_##NAME##_##OP##_reduce_on_stream(nvshmem_team_t team, TYPE *dest,                \
                                                  const TYPE *src, size_t nreduce,                \
                                                  nvshmemx_stream_t s) {                          \
        return reduce_on_stream(NVSHMEMI_DT_##TAG, NVSHMEMI_OP_##OP, team, dest, src, nreduce,    \
                                (hipStream_t)s);                                                  \
    }                                                                                             \
    int nvshmem_##NAME##_##OP##_reduce(nvshmem_team_t team, TYPE *dest, const TYPE *src,          \
                                       size_t nreduce) {                                          \
        return finish_blocking(reduce_on_stream(NVSHMEMI_DT_##TAG, NVSHMEMI_OP_##OP, team, dest,  \
                                                src, nreduce, nullptr));                          \
    }                                                                                             \
    int nvshmemx_##NAME##_##OP##_reducescatter_on_stream(nvshmem_team_t team, TYPE *dest,         \
                                                         const TYPE *src, size_t nreduce,         \
                                                         nvshmemx_stream_t s) {                   \
        return reducescatter_on_stream(NVSHMEMI_DT_##TAG, NVSHMEMI_OP_##OP, team, dest, src,      \
                                       nreduce, (hipStream_t)s);                                  \
    }                                                                                             \
    int nvshmem_##NAME##_##OP##_reducescatter(nvshmem_team_t team, TYPE *dest, const TYPE *src,   \
                                              size_t nreduce) {                                   \
        return finish_blocking(reducescatter_on_stream(NVSHMEMI_DT_##TAG, NVSHMEMI_OP_##OP, team, \
                                                       dest, src, nreduce, nullptr));             \
    }
NVSHMEMI_REPT_FOR_ALL_REDUCE_TYPES_AND_OPS(NVSHMEMI_DEFINE_TYPED_REDUCE_HOST)
#undef NVSHMEMI_DEFINE_TYPED_REDUCE_HOST

}  // extern "C"
