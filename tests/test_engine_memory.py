"""The engine where pinned or device memory is short (no GPU): the library on
a host model of the HIP allocation calls (tests/host/engine_memory.cpp)."""
import os
import subprocess

from pastix_amd import pastix

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_short_memory(tmp_path):
    exe = str(tmp_path / "engine_memory")
    lib = os.path.dirname(pastix.LIBPATH)
    subprocess.run(["g++", "-std=c++17", "-O1", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "pastix_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", "engine_memory.cpp"), "-o", exe, pastix.LIBPATH,
                    "-Wl,-rpath," + lib, "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib"], check=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0 and "0 failures" in p.stdout, (p.returncode, p.stdout, p.stderr)
