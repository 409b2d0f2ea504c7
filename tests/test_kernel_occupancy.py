"""Wavefronts per SIMD of the kernels that call the device API.  A collective launch takes no more blocks than are resident
together, so a copy or a fold that costs its callers registers makes launches fail that worked; and everything else in such
a kernel runs with fewer wavefronts to hide its latency."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIBRARY = os.path.join(ROOT, "nvshmem_amd", "lib", "libnvshmem_amd_perftest.so")
LLVM = "/opt/rocm/llvm/bin/"
THREAD, WARP, BLOCK = 0, 1, 2


@pytest.fixture(scope="module")
def registers(tmp_path_factory):
    """Vector registers of every kernel of the library, by mangled name."""
    d = tmp_path_factory.mktemp("code")
    fat = str(d / "fatbin")
    subprocess.run([LLVM + "llvm-objcopy", "--dump-section", ".hip_fatbin=" + fat, LIBRARY, str(d / "rest")], check=True)
    data = open(fat, "rb").read()
    found = {}
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        at = m.end() + 8
        for _ in range(struct.unpack_from("<Q", data, m.end())[0]):
            offset, size, name_len = struct.unpack_from("<QQQ", data, at)
            name = data[at + 24:at + 24 + name_len]
            at += 24 + name_len
            if b"gfx950" in name and size:
                unit = str(d / "unit.elf")
                open(unit, "wb").write(data[m.start() + offset:m.start() + offset + size])
                notes = subprocess.run([LLVM + "llvm-readelf", "--notes", unit], check=True, stdout=subprocess.PIPE, text=True).stdout
                for entry in re.split(r"\n\s+- \.agpr_count:", notes)[1:]:
                    found[re.search(r"\.symbol:\s+'?(\S+?)\.kd", entry).group(1)] = \
                        int(re.search(r"\.vgpr_count:\s+(\d+)", entry).group(1))
    assert found
    return found


def _wavefronts(registers, kernel):
    counts = [n for name, n in registers.items() if re.search(r"\d" + kernel, name)]
    assert counts, "no kernel " + kernel
    # 512 registers a lane and SIMD, dealt out in eights, and at most eight wavefronts
    return min(min(8, 512 // max(8, -(-n // 8) * 8)) for n in counts)


@pytest.mark.parametrize("kernel,least", [
    ("ring_reduce_kernelE", 7), ("pt2pt_latency_kernelE", 8), ("pingpong_kernelE", 8),
    ("ring_rma_kernelILi%dE" % WARP, 8), ("ring_rma_kernelILi%dE" % BLOCK, 8),
    ("put_signal_stream_kernelILi%dE" % WARP, 5), ("put_signal_stream_kernelILi%dE" % BLOCK, 7),
    ("alltoall_kernelILi%dE" % WARP, 7), ("alltoall_kernelILi%dE" % BLOCK, 8),
    ("fcollect_kernelILi%dE" % WARP, 7), ("fcollect_kernelILi%dE" % BLOCK, 8),
    ("broadcast_kernelILi%dE" % WARP, 8), ("broadcast_kernelILi%dE" % BLOCK, 8),
    ("team_coll_kernelILi%dE" % WARP, 5), ("team_coll_kernelILi%dE" % BLOCK, 4),
    ("moe_dispatch_kernelILb1E", 5), ("moe_dispatch_rowsignal_kernelILb1E", 4), ("moe_combine_kernelILb1E", 8)])
def test_callers_of_the_copy_engine(registers, kernel, least):
    assert _wavefronts(registers, kernel) >= least


@pytest.mark.parametrize("kernel,least", [("reduce_float_sum_kernel", 8), ("reduce_float_max_kernel", 8),
                                          ("reduce_int32_sum_kernel", 8), ("reduce_int64_xor_kernel", 8),
                                          ("reduce_uint64_and_kernel", 8), ("reduce_double_prod_kernel", 8),
                                          ("reduce_int16_min_kernel", 8), ("reduce_bfloat16_sum_kernel", 8),
                                          ("reduce_bfloat16_max_kernel", 7)])
def test_in_kernel_allreduce(registers, kernel, least):
    for scope in (THREAD, WARP, BLOCK):
        assert _wavefronts(registers, kernel + "ILi%dE" % scope) >= least
