"""The FP64 stage's unchecked quotients (vh::DivTry,
cpu-vh_amd/csrc/vh_device.hpp): over the exponents of numerator and divisor,
subnormal numerators and quotients included, whatever the policy's one check
accepts is the division operator's value bit for bit, and ordinary operands
and every quotient by 3 and 5 are accepted.  tests/divtry_check.cpp is compiled from the library's header for
the host, where the reciprocal is the correctly rounded one."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_accepted_quotients_are_the_operators(tmp_path):
    exe = str(tmp_path / "divtry_check")
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-host-only", "-O2", "-std=c++17", "-ffp-contract=off", "-mfma",
                    "-o", exe, os.path.join(HERE, "divtry_check.cpp")], check=True, capture_output=True)
    r = subprocess.run([exe, "2000000"], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and r.stdout.count("mismatches 0") == 11, r.stdout
