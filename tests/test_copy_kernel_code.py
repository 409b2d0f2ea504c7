"""What the compiler made of kernels for small messages: those that take a few microseconds are bound by the memory round
trips a wavefront makes one after the other, and these can be read from the loads and waits in its code."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIBRARY = os.path.join(ROOT, "nvshmem_amd", "lib", "libnvshmem_amd.so")
LLVM = "/opt/rocm/llvm/bin/"
MODES = {"fcollect": 0, "alltoall": 1, "broadcast": 2}
STREAMED = 2  # the store form of all three


PERFTEST = os.path.join(ROOT, "nvshmem_amd", "lib", "libnvshmem_amd_perftest.so")


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    """The GPU code of the library, one ELF file per translation unit."""
    return _units(LIBRARY, tmp_path_factory.mktemp("code"))


@pytest.fixture(scope="module")
def perftest_objects(tmp_path_factory):
    return _units(PERFTEST, tmp_path_factory.mktemp("perftest"))


def _units(library, d):
    fat = str(d / "fatbin")
    subprocess.run([LLVM + "llvm-objcopy", "--dump-section", ".hip_fatbin=" + fat, library, str(d / "rest")], check=True)
    data = open(fat, "rb").read()
    out = []
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        at = m.end()
        count, = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(count):
            offset, size, name_len = struct.unpack_from("<QQQ", data, at)
            name = data[at + 24:at + 24 + name_len]
            at += 24 + name_len
            if b"gfx950" in name and size:
                out.append(str(d / ("unit%d.elf" % len(out))))
                open(out[-1], "wb").write(data[m.start() + offset:m.start() + offset + size])
    assert out
    return out


def _kernel(code_objects, mode, streamed_loads=False, paced=False):
    """Instructions of one segment_copy_kernel, in the order in which they are laid out."""
    return _code(code_objects, r"segment_copy_kernelILi%dELb%dELb%dELi%dE" % (MODES[mode], streamed_loads, paced, STREAMED))


def _code(code_objects, kernel):
    symbol = re.compile(kernel)
    for path in code_objects:
        names = subprocess.run([LLVM + "llvm-objdump", "-t", path], check=True, stdout=subprocess.PIPE, text=True).stdout.split()
        for name in names:
            if symbol.search(name) and re.fullmatch(r"\w+", name):
                text = subprocess.run([LLVM + "llvm-objdump", "-d", "--no-show-raw-insn", "--disassemble-symbols=" + name, path],
                                      check=True, stdout=subprocess.PIPE, text=True).stdout
                return [line.split("//")[0].strip() for line in text.splitlines() if line.startswith("\t")]
    raise AssertionError("no kernel " + kernel)


def _places(code, what):
    return [i for i, line in enumerate(code) if re.match(what, line)]


@pytest.mark.parametrize("mode", sorted(MODES))
def test_edge_bytes_wait_beside_the_vectors(code_objects, mode):
    """The bytes around the vectors are stored after the vectors' load has gone out, not in a round trip before it."""
    code = _kernel(code_objects, mode)
    load, = _places(code, r"global_load_dwordx4")
    assert min(_places(code, r"global_store_byte")) > load


@pytest.mark.parametrize("mode", ["fcollect", "broadcast"])
def test_stores_to_several_members_do_not_wait(code_objects, mode):
    """Back to back: the loads are waited for once, and no wait stands between the stores (or in their loops)."""
    code = _kernel(code_objects, mode)
    first = min(_places(code, r"global_store_dwordx4"))
    assert not [i for i in _places(code, r"s_waitcnt.*vmcnt") if i > first]


@pytest.mark.parametrize("kernel", ["reduce_gather_kernelIfLi5ELi0ELb0ELb0E", "reducescatter_gather_kernelIfLi5ELi0ELb0E"])
def test_edge_elements_of_many_members_are_loaded_together(code_objects, kernel):
    """Teams whose size is not known at compile time: the elements around the vectors, one word each, are fetched from
    eight members at a time, without a wait between the loads."""
    code = _code(code_objects, kernel)
    longest = run = 0
    for line in code:
        if re.match(r"global_load_dword ", line):
            run += 1
            longest = max(longest, run)
        elif re.match(r"s_waitcnt.*vmcnt", line):
            run = 0
    assert longest >= 8


@pytest.mark.parametrize("kernel", [r"segment_copy_kernel", r"reduce_gather_kernel", r"reduce_element_kernel",
                                    r"reducescatter_gather_kernel", r"put_signal_kernel", r"strided_copy_kernel",
                                    r"signal_op_kernel", r"signal_wait_kernel", r"wait_until_kernel",
                                    r"wait_until_all_kernel", r"wait_until_all_vector_kernel", r"scalar_p_kernel"])
def test_kernels_of_small_calls_have_no_implicit_arguments(code_objects, kernel):
    """The host fills in a kernel's implicit arguments on every launch, which costs it a quarter of the launch."""
    seen = 0
    for path in code_objects:
        notes = subprocess.run([LLVM + "llvm-readelf", "--notes", path], check=True, stdout=subprocess.PIPE, text=True).stdout
        for entry in re.split(r"\n\s+- \.agpr_count:", notes)[1:]:
            if re.search(r"\.symbol:\s+\S*\d%s[IEP]\S*\.kd" % kernel, entry):
                seen += 1
                assert "hidden_" not in entry
    assert seen


def test_rows_of_a_full_size_dispatch_are_spaced(perftest_objects):
    """Long rows of much data: a wavefront asks for the row's place when the PE has arrived, behind a branch that others take."""
    code = _code(perftest_objects, r"moe_dispatch_kernelILb1E")
    places = _places(code, r"global_load_dwordx2")
    spaced = [i for i in places if [j for j in _places(code, r"global_load_dword ") if i - 16 < j < i]]
    assert spaced
    between = code[[j for j in _places(code, r"global_load_dword ") if j < spaced[0]][-1] + 1:spaced[0]]
    wait = [i for i, line in enumerate(between) if re.match(r"s_waitcnt.*vmcnt\(0\)", line)]
    assert wait and any(re.match(r"s_cbranch", line) for line in between[:wait[0]])


@pytest.mark.parametrize("full,outstanding", [(1, 2), (0, 13)])
def test_stores_of_long_rows_with_a_signal(perftest_objects, full, outstanding):
    """Fourteen write-through stores: in a full-size dispatch each from the fourth on waits until two are left, otherwise
    each waits for its own load alone."""
    code = _code(perftest_objects, r"moe_dispatch_rowsignal_kernelILb1ELb%dE" % full)
    runs, waits = [], 15
    for line in code:
        count = re.match(r"s_waitcnt.*vmcnt\((\d+)\)", line)
        if count:
            waits = min(waits, int(count.group(1)))
        elif line.startswith("buffer_load_dwordx4"):
            runs.append([])
        elif line.startswith("buffer_store_dwordx4") and " sc1" in line:
            runs[-1].append(waits)
            waits = 15
    longest = max(runs, key=len)
    assert len(longest) == 14 and set(longest[3:]) == {outstanding}
    for run in runs:
        assert 8 < len(run) or all(w >= len(run) - 1 for w in run[1:])
