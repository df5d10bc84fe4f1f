"""The stage derivatives of the quad form (solaris_amd/csrc/quad_stages.h),
checked on the host: every write stays inside the columns that are allotted
(tests/cpp/quad_stages_check.cpp, built with g++)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_quad_stages_host_check(tmp_path):
    exe = tmp_path / "quad_stages_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wno-unknown-pragmas", "-o", str(exe),
                    os.path.join(HERE, "cpp", "quad_stages_check.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "quad stages: ok" in r.stdout
