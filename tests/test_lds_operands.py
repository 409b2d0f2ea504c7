"""A put from LDS or a get into LDS must not go through buffer instructions: their descriptors reach global memory only, and
hold too few bits of the address to tell the two apart.  Compile only - no GPU is needed."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
HEADERS = '#include <hip/hip_runtime.h>\n#include "nvshmem.h"\n#include "nvshmemx.h"\n'
VISIBLE = HEADERS + """
__global__ void probe(char *p, size_t n, unsigned long long *out) {
    __shared__ __align__(16) char tile[8192];
    tile[threadIdx.x] = (char)n;
    __syncthreads();
    %s;
    __syncthreads();
    out[threadIdx.x] = tile[n];
}
"""
HIDDEN = HEADERS + """
__device__ __attribute__((noinline)) void copy(char *dst, const char *src, size_t n, uint64_t *sig, int pe) { %s; }
__global__ void probe(char **p, size_t n, uint64_t *sig) { copy(p[0], p[1], n, sig, 1); }
"""
PUT = "nvshmemi_memcpy_threadgroup<NVSHMEMI_THREADGROUP_WARP>(%s, %s, n)"
GET = "nvshmemi_memcpy_threadgroup<NVSHMEMI_THREADGROUP_WARP, NVSHMEMI_AMD_STORE_STREAM, NVSHMEMI_AMD_LOAD_STREAM>(%s, %s, n)"


def _compile(tmp_path, source):
    (tmp_path / "probe.hip").write_text(source)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-std=c++17", "-O3", "--cuda-device-only", "-S", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-I", os.path.join(ROOT, "include"), str(tmp_path / "probe.hip"), "-o",
                    str(tmp_path / "probe.asm")], check=True, timeout=600)
    return (tmp_path / "probe.asm").read_text()


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is not installed")
@pytest.mark.parametrize("copy,buffers", [(PUT % ("p", "tile + n % 16"), False), (GET % ("tile + n % 16", "p"), False),
                                          (PUT % ("p", "p + 65536"), True)], ids=["put", "get", "neither"])
def test_copies_that_the_compiler_sees_are_of_lds(tmp_path, copy, buffers):
    code = _compile(tmp_path, VISIBLE % copy)
    assert bool(re.search(r"buffer_(load|store)_dwordx4", code)) == buffers
    assert buffers or re.search(r"ds_(read|write)", code)


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is not installed")
@pytest.mark.parametrize("call", ["nvshmemx_putmem_warp(dst, src, n, pe)", "nvshmemx_getmem_warp(dst, src, n, pe)",
                                  "nvshmemx_putmem_signal_warp(dst, src, n, sig, 1, NVSHMEM_SIGNAL_ADD, pe)"])
def test_copies_of_any_address_compare_it_with_the_apertures(tmp_path, call):
    """There is no LDS here that a pointer could be made of: the apertures are named by the comparisons alone."""
    code = _compile(tmp_path, HIDDEN % call)
    assert "buffer_load_dwordx4" in code and "buffer_store_dwordx4" in code
    first = code.index("buffer_load_dwordx4")
    assert "src_shared_base" in code[:first] and "src_private_base" in code[:first]
