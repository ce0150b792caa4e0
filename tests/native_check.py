"""Builds a C++ check of the library's host code and runs it."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "argweaver_amd")
CSRC = os.path.join(PKG, "csrc")


def run_check(tmp_path, name, library=False):
    """tests/native/<name>.cpp; library: linked with the library, which then calls
    the check's fake_hip.h in the HIP runtime's place."""
    exe = str(tmp_path / name)
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-I" + CSRC,
           os.path.join(HERE, "native", name + ".cpp"), "-o", exe]
    if library:
        cmd += ["-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-Wno-unused-result",
                "-rdynamic", "-Wl,--allow-shlib-undefined", "-Wl,-rpath," + PKG,
                os.path.join(PKG, "libargweaver_amd.so")]
    subprocess.check_call(cmd)
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=60)
    assert r.returncode == 0, r.stdout.decode()
