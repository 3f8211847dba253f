"""Overlapping vh_fo_flag_noalloc calls share their scratch: whatever each
reads there, the ids it writes stay within its array and its lattice
(vh::fo_flag_place, cpu-vh_amd/csrc/vh_kernels.hpp, with the scratch laid out as
vh_noalloc.hip lays it out).  tests/flag_overlap_check.cpp runs the passes'
blocks of two calls in random order on the host."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_overlapping_calls_stay_in_bounds(tmp_path):
    exe = str(tmp_path / "flag_overlap_check")
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-host-only", "-O2", "-std=c++17", "-o", exe,
                    os.path.join(HERE, "flag_overlap_check.cpp")], check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and r.stdout.strip() == "cases 3840 bad 0", r.stdout
