"""Builds a C++ check of the library's host code and runs it."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "argweaver_amd", "csrc")


def run_check(tmp_path, name, sources=(), flags=()):
    exe = str(tmp_path / name)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-I" + CSRC] +
                          list(flags) + [os.path.join(HERE, "native", name + ".cpp")] +
                          [os.path.join(CSRC, s) for s in sources] + ["-o", exe])
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=60)
    assert r.returncode == 0, r.stdout.decode()
