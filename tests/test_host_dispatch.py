"""The engine's dispatch, graphs and memory limits on the CPU (see host_dispatch.py): every check runs in
a process of its own on a HIP runtime without a device."""
import os
import subprocess
import sys

import pytest

import host_dispatch

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("runtime") / "libhostruntime.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "host_runtime.cpp"), "-o", lib], check=True)
    return lib


@pytest.mark.parametrize("name", sorted(host_dispatch.CHECKS))
def test_dispatch(runtime, name):
    r = subprocess.run([sys.executable, os.path.join(HERE, "host_dispatch.py"), runtime, name], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
