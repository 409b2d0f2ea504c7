"""Runs a piece of a test in a process of its own where the library's launches are recorded instead of run."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes as C, os, sys
sys.path.insert(0, %(root)r)
recorder = C.CDLL(%(recorder)r, mode=C.RTLD_GLOBAL)
recorder.recorder_kernel.restype = C.c_char_p
from nvshmem_amd import _lib
lib = _lib.load()

def launches():
    '''What has been launched since the last call: (kernel, cooperative, grid, block, dynamic LDS).'''
    out, v = [], (C.c_ulonglong * 8)()
    for i in range(recorder.recorder_count()):
        recorder.recorder_shape(i, v)
        out.append((recorder.recorder_kernel(i).decode(), bool(v[0]), tuple(v[1:4]), tuple(v[4:7]), v[7]))
    recorder.recorder_clear()
    return out

def ok(rc):
    assert rc == 0, lib.nvshmemx_amd_last_error().decode()
"""


@pytest.fixture(scope="session")
def recorded(tmp_path_factory):
    """recorded(code, **environment) runs `code` behind the prelude above."""
    so = str(tmp_path_factory.mktemp("recorder") / "liblaunch_recorder.so")
    build = subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                            os.path.join(ROOT, "tests", "native", "launch_recorder.cpp"), "-o", so],
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert build.returncode == 0, build.stdout

    def run(code, **environment):
        env = {k: v for k, v in os.environ.items() if not k.startswith("NVSHMEM_")}
        env.update(environment)
        done = subprocess.run([sys.executable, "-c", PRELUDE % {"root": ROOT, "recorder": so} + code], env=env,
                              stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
        assert done.returncode == 0, done.stdout
        return done.stdout

    return run
