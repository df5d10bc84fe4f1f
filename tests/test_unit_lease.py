"""The leases of compute units (solaris_amd/csrc/unit_lease.h), checked on the
host (tests/cpp/unit_lease_check.cpp, built with g++)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_unit_lease_host_check(tmp_path):
    exe = tmp_path / "unit_lease_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-o", str(exe),
                    os.path.join(HERE, "cpp", "unit_lease_check.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "unit leases: ok" in r.stdout
