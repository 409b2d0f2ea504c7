"""The measured work of this library: what a program that uses it has it do, through its public entry points.

A program of this library keeps its tensors in the symmetric heap (one slice per logical PE on one GPU), keeps
its bound entry points and addresses, and calls collectives, host-initiated RMA, its own device-API kernels
and the token shuffle on the stream that its other work is on.  The kinds of work below are

  allreduce, reducescatter, fcollect, alltoall, broadcast   host-launched collectives on a stream
  ring         every PE puts to / gets from its neighbour inside a kernel (block-scoped RMA)
  inkernel     a collective that a kernel calls in the middle of its own work, one block per PE
  moe          token shuffle: dispatch with a signal per row, then combine
  halo         2-D halo exchange by host-initiated RMA: rows with put_signal, columns with iput

All of them return whole results: the destination on every PE.
"""
import ctypes as C
import math

import torch

from nvshmem_amd import _lib

TEAM_WORLD = 0
SCOPE_WARP, SCOPE_BLOCK = 1, 2
SIGNAL_ADD, CMP_GE = 10, 5
PER_ROW_PAYLOAD_ORDER = SCOPE_WARP | 256 | 512  # nvshmem_perftest_moe_dispatch_put_signal: a payload-only signal per row

HEAP_BYTES = 64 << 30  # of all PEs together
MiB = 1 << 20

# API type -> (torch dtype, storage type of __cuda_array_interface__, element kind of the device collectives)
TYPES = {
    "float": (torch.float32, "<f4", 10), "double": (torch.float64, "<f8", 11),
    "bfloat16": (torch.bfloat16, "<i2", 9), "half": (torch.float16, "<f2", 8),
    "int32": (torch.int32, "<i4", 2), "int64": (torch.int64, "<i8", 3), "uint8": (torch.uint8, "|u1", 4),
}
OPS = {"xor": 2, "max": 4, "sum": 5}


def listed():
    return [
        # a norm, a loss, a handful of statistics: the smallest allreduce, all latency
        {"name": "allreduce_f32_8KiB", "kind": "allreduce", "npes": 8, "type": "float", "op": "sum", "n": 2048,
         "dst_shift": 0, "src_shift": 0},
        # one 25 MiB gradient bucket inside a flat buffer: it starts and ends where the parameters do
        {"name": "allreduce_bf16_bucket", "kind": "allreduce", "npes": 8, "type": "bfloat16", "op": "sum",
         "n": 13107203, "dst_shift": 3, "src_shift": 3},
        # the largest: 256 MiB of fp32 on every PE
        {"name": "allreduce_f32_256MiB", "kind": "allreduce", "npes": 8, "type": "float", "op": "sum", "n": 1 << 26,
         "dst_shift": 0, "src_shift": 0},
        # sharded data parallelism: gradients to their owners, parameters back to everybody.  The flat parameter is
        # padded to a multiple of the PE count only, so a shard is an odd number of elements.
        {"name": "reducescatter_bf16_shard", "kind": "reducescatter", "npes": 8, "type": "bfloat16", "op": "sum",
         "n": 1500007, "dst_shift": 0, "src_shift": 0},
        {"name": "fcollect_bf16_shard", "kind": "fcollect", "npes": 8, "type": "bfloat16", "n": 1500007,
         "dst_shift": 0, "src_shift": 0},
        # a transposition between two decompositions of one array, 16 PEs, a few KiB for each of the others
        {"name": "alltoall_f32_16KiB", "kind": "alltoall", "npes": 16, "type": "float", "n": 4093, "dst_shift": 0,
         "src_shift": 0},
        # weights or a table from one PE to all
        {"name": "broadcast_32MiB", "kind": "broadcast", "npes": 8, "type": "uint8", "n": 33554437, "root": 3,
         "dst_shift": 0, "src_shift": 0},
        # the library's headline: the neighbour put of the put bandwidth test at its largest size and launch shape
        {"name": "ring_put_256MiB", "kind": "ring", "npes": 8, "get": False, "n": 256 * MiB, "blocks": 16,
         "threads": 1024, "dst_shift": 0, "src_shift": 0},
        # partial sums of 16 rows of 7168 bf16 added up inside the kernel that made them
        {"name": "inkernel_allreduce_bf16", "kind": "inkernel", "npes": 8, "type": "bfloat16", "op": "sum",
         "n": 16 * 7168, "threads": 1024},
        # token shuffle, decode and prefill: rows of 7168 bf16, top-8 of 256 experts
        {"name": "moe_decode", "kind": "moe", "npes": 8, "tokens": 64, "topk": 8, "experts": 256, "row": 14336},
        {"name": "moe_prefill", "kind": "moe", "npes": 8, "tokens": 4096, "topk": 8, "experts": 256, "row": 14336},
        # a stencil's tiles on a 2 x 4 grid of PEs, one cell of halo, periodic
        {"name": "halo_f32_2048", "kind": "halo", "npes": 8, "type": "float", "rows": 2048, "cols": 2048},
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["allreduce", "allreduce", "reducescatter", "fcollect", "alltoall", "broadcast", "ring",
                       "inkernel", "moe", "halo"])
    npes = rng.choice([4, 8, 8, 16])
    # half of the buffers start on an allocation's boundary, half at some element of a larger buffer
    shifts = {"dst_shift": 0, "src_shift": 0} if rng.random() < 0.5 else \
             {"dst_shift": rng.randrange(16), "src_shift": rng.randrange(16)}
    if kind in ("allreduce", "reducescatter"):
        t, op = rng.choice([("float", "sum"), ("float", "max"), ("bfloat16", "sum"), ("bfloat16", "max"),
                            ("half", "sum"), ("double", "sum"), ("int32", "sum"), ("int64", "xor")])
        es = _size(t)
        # bytes of source per PE
        n = _spread(rng, 512, 64 * MiB) // es // (npes if kind == "reducescatter" else 1) + 1
        return dict({"kind": kind, "npes": npes, "type": t, "op": op, "n": _ragged(rng, n)}, **shifts)
    if kind in ("fcollect", "alltoall"):
        t = rng.choice(["float", "bfloat16", "int64", "uint8"])
        # bytes of a segment: npes of them arrive on every PE
        n = _spread(rng, 64, 16 * MiB * 8 // npes) // _size(t) + 1
        return dict({"kind": kind, "npes": npes, "type": t, "n": _ragged(rng, n)}, **shifts)
    if kind == "broadcast":
        return dict({"kind": kind, "npes": npes, "type": "uint8", "n": _ragged(rng, _spread(rng, 256, 256 * MiB)),
                     "root": rng.randrange(npes)}, **shifts)
    if kind == "ring":
        blocks = rng.choice([1, 4, 16])
        return dict({"kind": kind, "npes": 8, "get": rng.random() < 0.5,
                     "n": _ragged(rng, _spread(rng, 1024, blocks * 16 * MiB)), "blocks": blocks,
                     "threads": rng.choice([256, 512, 1024])}, **shifts)
    if kind == "inkernel":
        t, op = rng.choice([("float", "sum"), ("float", "max"), ("bfloat16", "sum"), ("bfloat16", "max")])
        return {"kind": kind, "npes": npes, "type": t, "op": op, "n": _ragged(rng, _spread(rng, 64, 1 << 20)),
                "threads": rng.choice([256, 512, 1024])}
    if kind == "moe":
        return {"kind": kind, "npes": 8, "tokens": _spread(rng, 8, 4096), "topk": rng.choice([2, 4, 6, 8]),
                "experts": rng.choice([64, 128, 256]), "row": 256 * rng.randrange(8, 57)}
    return {"kind": "halo", "npes": npes, "type": rng.choice(["float", "double"]), "rows": _spread(rng, 64, 4096),
            "cols": _spread(rng, 64, 4096)}


def _ragged(rng, n):
    """Every second size is rounded up to a multiple of 64 elements, the others stay as they fell."""
    return n if rng.random() < 0.5 else (n + 63) // 64 * 64


def _size(type_name):
    return torch.empty(0, dtype=TYPES[type_name][0]).element_size()


# ------------------------------------------------------------------------------------------------------------
# The symmetric heap, as tensors
# ------------------------------------------------------------------------------------------------------------
_live = 0  # objects that hold memory of the current heap


def _heap(npes):
    """The library, initialised for npes PEs: a heap that nothing holds memory of makes room for one of another PE count."""
    lib = _lib.load()
    if lib.nvshmem_n_pes() != npes or not lib.nvshmemx_init_status():
        if _live:
            raise RuntimeError("symmetric memory of %d PEs is still in use" % lib.nvshmem_n_pes())
        torch.cuda.synchronize()
        lib.nvshmem_finalize()
        rc = lib.nvshmemx_amd_init(npes, HEAP_BYTES // npes)
        if rc != 0:
            raise RuntimeError("nvshmemx_amd_init: %s" % lib.nvshmemx_amd_last_error().decode())
    return lib


class _Memory:
    """One symmetric allocation."""

    def __init__(self, lib, nbytes):
        global _live
        self.lib, self.address = lib, lib.nvshmem_malloc(max(nbytes, 16))
        if not self.address:
            raise MemoryError("out of memory: %d bytes per PE" % nbytes)
        _live += 1
        self.stride = lib.nvshmem_ptr(self.address, 1) - lib.nvshmem_ptr(self.address, 0)

    def __del__(self):
        global _live
        if getattr(self, "address", None):
            self.lib.nvshmem_free(self.address)
            self.address = None
            _live -= 1


class _Exposed:
    def __init__(self, memory, interface):
        self.memory, self.__cuda_array_interface__ = memory, interface  # a tensor keeps this object, and so the memory


def _tensor(memory, type_name, shape, first=0, npes=None):
    """[npes, *shape] tensor over every PE's copy, from element `first` of the allocation on."""
    dtype, storage, _ = TYPES[type_name]
    es = _size(type_name)
    strides, step = [], es
    for extent in reversed(shape):
        strides.insert(0, step)
        step *= extent
    count = npes or memory.lib.nvshmem_n_pes()
    view = torch.as_tensor(_Exposed(memory, {
        "shape": (count,) + tuple(shape), "typestr": storage, "version": 3, "strides": (memory.stride,) + tuple(strides),
        "data": (memory.lib.nvshmem_ptr(memory.address, 0) + first * es, False)}), device="cuda")
    return view.view(dtype)


def _fill(tensors, seed):
    """Activations and gradients: normal.  Whole numbers and bytes: all values."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    for t in tensors:
        for pe in range(t.shape[0]):
            if t.dtype.is_floating_point:
                t[pe].normal_(generator=g)
            else:
                info = torch.iinfo(t.dtype)
                t[pe].random_(info.min, info.max, generator=g)


class _State:
    """What a program keeps: its buffers, and its calls with their arguments."""

    def __init__(self):
        self.calls, self.outputs, self.keep = [], [], []


def _call(state, fn, *args):
    state.calls.append((fn, args))


def _bind(lib, name, argtypes, restype=C.c_int):
    fn = getattr(lib, name)
    fn.argtypes, fn.restype = argtypes, restype
    return fn


_vp, _sz, _i32, _u64, _pd = C.c_void_p, C.c_size_t, C.c_int, C.c_uint64, C.c_ssize_t


# ------------------------------------------------------------------------------------------------------------
# prepare
# ------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    state = _State()
    lib = _heap(case["npes"])
    stream = torch.cuda.current_stream().cuda_stream or None
    PREPARE[case["kind"]](case, seed, state, lib, stream)
    return state


def _buffers(case, state, lib, seed, dst_elems, src_elems):
    es = _size(case["type"])
    src = _Memory(lib, (src_elems + case.get("src_shift", 0)) * es)
    dst = _Memory(lib, (dst_elems + case.get("dst_shift", 0)) * es)
    _fill([_tensor(src, case["type"], (src_elems,), case.get("src_shift", 0))], seed)
    out = _tensor(dst, case["type"], (dst_elems,), case.get("dst_shift", 0))
    out.zero_()
    state.keep += [src, dst]
    state.outputs.append(out)
    return dst.address + case.get("dst_shift", 0) * es, src.address + case.get("src_shift", 0) * es


def _prepare_reduction(case, seed, state, lib, stream):
    scatter = case["kind"] == "reducescatter"
    dst, src = _buffers(case, state, lib, seed, case["n"], case["n"] * (case["npes"] if scatter else 1))
    fn = _lib.typed_coll(lib, "nvshmemx_%s_%s_%s_on_stream" % (case["type"], case["op"], "reducescatter" if scatter else "reduce"), True)
    _call(state, fn, TEAM_WORLD, dst, src, case["n"], stream)


def _prepare_collect(case, seed, state, lib, stream):
    n, npes = case["n"], case["npes"]
    dst, src = _buffers(case, state, lib, seed, n * npes, n * (npes if case["kind"] == "alltoall" else 1))
    fn = _lib.typed_coll(lib, "nvshmemx_%s_%s_on_stream" % (case["type"], case["kind"]), True)
    _call(state, fn, TEAM_WORLD, dst, src, n, stream)


def _prepare_broadcast(case, seed, state, lib, stream):
    dst, src = _buffers(case, state, lib, seed, case["n"], case["n"])
    _call(state, lib.nvshmemx_broadcastmem_on_stream, TEAM_WORLD, dst, src, case["n"], case["root"], stream)


def _prepare_ring(case, seed, state, lib, stream):
    dst, src = _buffers(dict(case, type="uint8"), state, lib, seed, case["n"], case["n"])
    if case["n"] % 4 == 0 and case["dst_shift"] % 4 == 0:  # the same bytes, in fewer values
        state.outputs = [_tensor(state.keep[1], "int32", (case["n"] // 4,), case["dst_shift"] // 4)]
    _call(state, _lib.load_perftest().nvshmem_perftest_ring_rma, dst, src, case["n"], case["blocks"], case["threads"],
          SCOPE_BLOCK, int(case["get"]), 1, stream)


def _prepare_inkernel(case, seed, state, lib, stream):
    dst, src = _buffers(case, state, lib, seed, case["n"], case["n"])
    _call(state, _lib.load_perftest().nvshmem_perftest_device_reduce, TYPES[case["type"]][2], OPS[case["op"]], dst, src,
          case["n"], SCOPE_BLOCK, case["threads"], stream)


def _route(case, seed):
    """Top-k distinct experts per token, the k-th most popular expert with probability ~ k^-1.1; the experts are dealt
    to the PEs in the order of their load, as a planner does that keeps the hottest ones apart: no PE gets more
    than its share of the copies and the hottest expert's, at most one a token.  Rows are grouped on the
    destination PE by (expert, source PE, token)."""
    npes, tokens, topk, experts = case["npes"], case["tokens"], case["topk"], case["experts"]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    gumbel = torch.empty(npes * tokens, experts, device="cuda").exponential_(generator=g).log_().neg_()
    popularity = torch.arange(1, experts + 1, device="cuda", dtype=torch.float32).log_().mul_(-1.1)
    chosen = (popularity + gumbel).topk(topk, dim=1).indices.reshape(npes, tokens * topk)
    loads = torch.bincount(chosen.reshape(-1), minlength=experts)
    rank = torch.empty_like(loads)
    rank[torch.sort(loads, descending=True, stable=True).indices] = torch.arange(experts, device="cuda")
    expert = (rank % npes * (experts // npes) + rank // npes)[chosen]
    pe = expert // (experts // npes)
    rows = torch.bincount(pe.reshape(-1), minlength=npes)
    source = torch.arange(npes, device="cuda").unsqueeze(1).expand_as(expert)
    order = torch.sort((expert * npes + source).reshape(-1), stable=True).indices
    place = torch.empty_like(order)
    place[order] = torch.arange(order.numel(), device="cuda")
    row = place.reshape(npes, -1) - (rows.cumsum(0) - rows)[pe]
    expected = torch.bincount((pe * npes + source).reshape(-1), minlength=npes * npes).reshape(npes, npes)
    return pe.to(torch.int32), row, expected


def _prepare_moe(case, seed, state, lib, stream):
    npes, tokens, topk, row = case["npes"], case["tokens"], case["topk"], case["row"]
    pe, at, expected = _route(case, seed)
    copies, cap, sig_stride = tokens * topk, tokens * (topk + npes), 16  # a 128-byte line per signal word
    send, recv, out = (_Memory(lib, n * row) for n in (tokens, cap, copies))
    d_pe, d_row, d_expected, sig = (_Memory(lib, n) for n in (4 * copies, 8 * copies, 8 * npes, 8 * npes * sig_stride))
    _fill([_tensor(send, "bfloat16", (tokens, row // 2))], seed + 1)
    _tensor(d_pe, "int32", (copies,)).copy_(pe)
    _tensor(d_row, "int64", (copies,)).copy_(at)
    _tensor(d_expected, "int64", (npes,)).copy_(expected)
    received = _tensor(recv, "bfloat16", (cap, row // 2))
    received.zero_()  # rows that nothing is sent to stay as they are
    state.keep += [send, recv, out, d_pe, d_row, d_expected, sig]
    state.outputs += [received, _tensor(out, "bfloat16", (copies, row // 2)), _tensor(sig, "int64", (npes * sig_stride,))]
    perf = _lib.load_perftest()
    _call(state, perf.nvshmem_perftest_fill_words, sig.address, 0, npes * sig_stride, stream)
    _call(state, perf.nvshmem_perftest_moe_dispatch_put_signal, recv.address, cap, send.address, d_pe.address, d_row.address,
          d_expected.address, sig.address, sig_stride, tokens, topk, row, 64, 256, PER_ROW_PAYLOAD_ORDER, stream)
    _call(state, perf.nvshmem_perftest_moe_combine_pieces, out.address, recv.address, cap, d_pe.address, d_row.address,
          tokens, topk, row, 2048, copies * ((row + 2047) // 2048), 64, SCOPE_WARP, stream)


def _grid(npes):
    return {4: (2, 2), 8: (2, 4), 16: (4, 4)}[npes]


def _prepare_halo(case, seed, state, lib, stream):
    npes, t, rows, cols = case["npes"], case["type"], case["rows"], case["cols"]
    es, width = _size(t), cols + 2
    tile, sig = _Memory(lib, (rows + 2) * width * es), _Memory(lib, 4 * 8)
    view, words = _tensor(tile, t, (rows + 2, width)), _tensor(sig, "int64", (4,))
    _fill([view], seed)
    words.zero_()
    state.keep += [tile, sig]
    state.outputs += [view, words]
    row = _bind(lib, "nvshmemx_%s_put_signal_on_stream" % t, [_vp, _vp, _sz, _vp, _u64, _i32, _i32, _vp], None)
    column = _bind(lib, "nvshmemx_%s_iput_on_stream" % t, [_vp, _vp, _pd, _pd, _sz, _i32, _vp], None)
    signal = lib.nvshmemx_signal_op_on_stream
    wait = _bind(lib, "nvshmemx_uint64_wait_until_all_on_stream", [_vp, _sz, _vp, _i32, _u64, _vp], None)
    down, right = _grid(npes)

    def cell(r, c):
        return (r * width + c) * es

    for pe in range(npes):
        y, x = divmod(pe, right)
        mine = lib.nvshmem_ptr(tile.address, pe)
        north, south = (y - 1) % down * right + x, (y + 1) % down * right + x
        west, east = y * right + (x - 1) % right, y * right + (x + 1) % right
        # my first row becomes the northern neighbour's lower halo, and so on round the tile
        _call(state, row, tile.address + cell(rows + 1, 1), mine + cell(1, 1), cols, sig.address, 1, SIGNAL_ADD, north, stream)
        _call(state, row, tile.address + cell(0, 1), mine + cell(rows, 1), cols, sig.address + 8, 1, SIGNAL_ADD, south, stream)
        _call(state, column, tile.address + cell(1, cols + 1), mine + cell(1, 1), width, width, rows, west, stream)
        _call(state, signal, sig.address + 16, 1, SIGNAL_ADD, west, stream)
        _call(state, column, tile.address + cell(1, 0), mine + cell(1, cols), width, width, rows, east, stream)
        _call(state, signal, sig.address + 24, 1, SIGNAL_ADD, east, stream)
    state.waits = [(wait, lib.nvshmem_ptr(sig.address, pe), stream) for pe in range(npes)]
    state.steps = 0


PREPARE = {"allreduce": _prepare_reduction, "reducescatter": _prepare_reduction, "fcollect": _prepare_collect,
           "alltoall": _prepare_collect, "broadcast": _prepare_broadcast, "ring": _prepare_ring,
           "inkernel": _prepare_inkernel, "moe": _prepare_moe, "halo": _prepare_halo}


# ------------------------------------------------------------------------------------------------------------
# run, work, tolerance
# ------------------------------------------------------------------------------------------------------------
def run(state):
    for fn, args in state.calls:
        if fn(*args):
            raise RuntimeError("%s: %s" % (fn.__name__, _lib.load().nvshmemx_amd_last_error().decode()))
    if hasattr(state, "waits"):
        state.steps += 1
        for wait, words, stream in state.waits:  # a PE computes on its tile when its four halos have come
            wait(words, 4, None, CMP_GE, state.steps, stream)
    return state.outputs


def work(case):
    kind, npes = case["kind"], case["npes"]
    if kind == "moe":
        rows = npes * case["tokens"] * case["topk"]
        # dispatch: a token's row read once, a copy per expert written; combine: every copy read and written
        return {"bytes": (npes * case["tokens"] + 3 * rows) * case["row"], "flops": 0}
    if kind == "halo":
        return {"bytes": 2 * npes * 2 * (case["rows"] + case["cols"]) * _size(case["type"]), "flops": 0}
    if kind == "ring":
        return {"bytes": 2 * npes * case["n"], "flops": 0}
    size = case["n"] * _size(case["type"])
    adds = {"allreduce": 1, "inkernel": 1, "reducescatter": npes}.get(kind, 0) * case["n"] * (npes - 1)
    moved = {"allreduce": 2 * npes, "inkernel": 2 * npes, "reducescatter": npes * npes + npes,
             "fcollect": npes + npes * npes, "alltoall": 2 * npes * npes, "broadcast": 1 + npes}[kind]
    return {"bytes": moved * size, "flops": adds}


def tolerance(case):
    """Everything but a floating-point sum is the same bits.  Sums: four times what adding the same eight normal
    values per element in the opposite order changes (rounded after every step, as the library's element-type
    arithmetic is)."""
    if case["kind"] not in ("allreduce", "reducescatter", "inkernel") or case["op"] != "sum":
        return "exact"
    return {"float": {"rel": 3.2e-7, "max": 1.8e-6}, "bfloat16": {"rel": 2.0e-2, "max": 0.11},
            "half": {"rel": 2.6e-3, "max": 1.3e-2}, "double": {"rel": 6e-16, "max": 3.6e-15}}.get(case["type"], "exact")
