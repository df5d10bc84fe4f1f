"""What the library asks of the HIP runtime, checked on the host: programs
that take the runtime's place (tests/cpp/fake_hip.h) count its calls."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "solaris_amd")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def run(tmp_path, name):
    if not os.path.exists(os.path.join(PKG, "libsolaris_amd.so")):
        pytest.skip("library not built")
    exe = tmp_path / name
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", "-rdynamic", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                    "-o", str(exe), os.path.join(HERE, "cpp", name + ".cpp"), f"-L{PKG}", "-lsolaris_amd",
                    f"-Wl,-rpath,{PKG}", f"-L{ROCM}/lib", f"-Wl,-rpath,{ROCM}/lib"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


def test_driver_calls(tmp_path):
    assert "driver calls: ok" in run(tmp_path, "driver_calls_check")


def test_context_calls(tmp_path):
    assert "context calls: ok" in run(tmp_path, "context_calls_check")


def test_error_calls(tmp_path):
    assert "error calls: ok" in run(tmp_path, "error_calls_check")


def test_ensemble_calls(tmp_path):
    assert "ensemble calls: ok" in run(tmp_path, "ensemble_calls_check")
