"""Builds the in-tree libraries.

  solaris_amd/libsolaris_amd.so   HIP kernels + the C ABI (hipcc, gfx950)
  solaris_amd/libsolaris_dropin.so  C++ classes with the reference's
                                    Acceleration / integrator / BodyData
                                    interfaces on top of the C ABI (g++)

Every HIP translation unit is compiled with packed FP32 instructions
disabled (-Xclang -target-feature -Xclang -packed-fp32-ops).
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
DROPIN = os.path.join(HERE, "dropin")
BUILD = os.path.join(ROOT, "_build")
LIB = os.path.join(HERE, "libsolaris_amd.so")
DROPIN_LIB = os.path.join(HERE, "libsolaris_dropin.so")

ARCH = os.environ.get("SOLARIS_AMD_ARCH", "gfx950")
HIPCC = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")
HIP_FLAGS = ["-O3", "-fPIC", "-std=c++17", f"--offload-arch={ARCH}",
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
             "-Wall", "-Wno-unused-function", "-Wno-unused-variable"]
HIP_SOURCES = ["pairs.hip", "stages.hip", "resident.hip", "mesh.hip", "quad.hip", "adjoint.hip", "adjoint_few.hip", "nngrid.hip", "noalloc.hip", "context.cpp",
               "ensemble.cpp", "adjoint.cpp"]


def _run(cmd, quiet=True):
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in p.stdout.splitlines()
                    if "packed-fp32-ops' is not a recognized feature" not in l)
    if p.returncode != 0:
        raise RuntimeError(f"build step failed ({p.returncode}): {' '.join(cmd)}\n{out}")
    if out.strip() and not quiet:
        print(out)
    return out


def build_hip(verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    objs = []
    cmds = []
    for src in HIP_SOURCES:
        obj = os.path.join(BUILD, src.replace(".", "_") + ".o")
        lang = ["-x", "hip"] if src.endswith(".hip") else []
        cmds.append([HIPCC, *HIP_FLAGS, *lang, "-c", os.path.join(CSRC, src), "-o", obj])
        objs.append(obj)
    with ThreadPoolExecutor(max_workers=min(8, len(cmds))) as ex:
        list(ex.map(lambda c: _run(c, not verbose), cmds))
    tmp = LIB + ".tmp"
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs], not verbose)
    os.replace(tmp, LIB)
    return LIB


def build_dropin(verbose: bool = False) -> str:
    """The drop-in classes (dropin/*.cpp) with the standalone definitions of
    the plain data classes (dropin/standalone/*.cpp, dropin/include/*.h),
    and the C++ driver program tests/cpp/dropin_driver."""
    srcs = sorted(os.path.join(DROPIN, f) for f in os.listdir(DROPIN) if f.endswith(".cpp"))
    std = os.path.join(DROPIN, "standalone")
    srcs += sorted(os.path.join(std, f) for f in os.listdir(std) if f.endswith(".cpp"))
    inc = [f"-I{os.path.join(DROPIN, 'include')}", f"-I{DROPIN}", f"-I{os.path.join(ROOT, 'include')}"]
    tmp = DROPIN_LIB + ".tmp"
    _run(["g++", "-O2", "-fPIC", "-shared", "-std=c++17", "-Wall", *inc, "-o", tmp, *srcs,
          f"-L{HERE}", "-lsolaris_amd", "-Wl,-rpath,$ORIGIN"], not verbose)
    os.replace(tmp, DROPIN_LIB)
    drv_src = os.path.join(ROOT, "tests", "cpp", "dropin_driver.cpp")
    if os.path.exists(drv_src):
        exe = os.path.join(ROOT, "tests", "cpp", "dropin_driver")
        _run(["g++", "-O2", "-std=c++17", "-Wall", *inc, "-o", exe + ".tmp", drv_src,
              f"-L{HERE}", "-lsolaris_dropin", "-lsolaris_amd", f"-Wl,-rpath,{HERE}"], not verbose)
        os.replace(exe + ".tmp", exe)
    return DROPIN_LIB


def build_host(verbose: bool = False) -> str:
    """solaris_amd/solaris_run: the scenario program (host/*.cpp, g++) over
    the C ABI of libsolaris_amd.so."""
    host = os.path.join(HERE, "host")
    srcs = sorted(os.path.join(host, f) for f in os.listdir(host) if f.endswith(".cpp"))
    exe = os.path.join(HERE, "solaris_run")
    _run(["g++", "-O2", "-std=c++17", "-Wall", "-ffp-contract=off", f"-I{os.path.join(ROOT, 'include')}",
          "-o", exe + ".tmp", *srcs, f"-L{HERE}", "-lsolaris_amd", "-Wl,-rpath,$ORIGIN"], not verbose)
    os.replace(exe + ".tmp", exe)
    return exe


def device_assembly(src: str) -> str:
    """gfx950 assembly of one HIP source of this library, compiled with the
    library's own flags (for inspection by the tests)."""
    out = os.path.join(BUILD, os.path.basename(src) + ".s")
    os.makedirs(BUILD, exist_ok=True)
    lang = ["-x", "hip"] if src.endswith(".hip") else []
    _run([HIPCC, *HIP_FLAGS, *lang, "--cuda-device-only", "-S", os.path.join(CSRC, src), "-o", out])
    with open(out) as f:
        return f.read()


def check_dropin_against(reference_include: str) -> None:
    """Compiles the drop-in set against another tree's headers (the
    reference's Solaris/ directory) to show the classes keep its
    interface."""
    for f in ("Acceleration", "RungeKuttaFehlberg78", "RungeKutta4", "DormandPrince", "dropin_bridge"):
        _run(["g++", "-std=c++11", "-fsyntax-only", "-fpermissive", "-w", "-include", "cstring",
              "-include", "cmath", "-include", "stdlib.h", f"-I{reference_include}", f"-I{DROPIN}",
              f"-I{os.path.join(ROOT, 'include')}", os.path.join(DROPIN, f + ".cpp")])


def build_all(verbose: bool = False):
    build_hip(verbose)
    build_dropin(verbose)
    build_host(verbose)


if __name__ == "__main__":
    build_all(verbose="-v" in sys.argv)
    print("built", LIB)
