"""Copies through pinned slots (nmesh_amd/csrc/host_copy.cpp) on the CPU, with
stand-ins for the HIP calls (host_copy_client.cpp): sizes around the slots' and
the thresholds, a queued copy that fails, and a machine without memory for more
threads, where those that run take all the chunks."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def client(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("hc") / "host_copy_client")
    src = os.path.join(HERE, "..", "nmesh_amd", "csrc", "host_copy.cpp")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", exe,
                           os.path.join(HERE, "host_copy_client.cpp"), src, "-pthread"])
    return exe


@pytest.mark.parametrize("what", ["round", "memcpy", "threads"])
def test_host_copy(client, what):
    p = subprocess.run([client, what], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, (p.returncode, p.stdout, p.stderr[-500:])
