"""Downloads and status reads of one owner from two threads (vh::HostCopy,
cpu-vh_amd/csrc/vh_hostcopy.hpp): each thread gets the error word its own copy
brought.  tests/hostcopy_check.cpp is built for the host, the HIP calls it needs
defined in it."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_status_of_another_thread_does_not_mix(tmp_path):
    exe = str(tmp_path / "hostcopy_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", exe,
                    os.path.join(HERE, "hostcopy_check.cpp")], check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
