"""Builds and runs a small C++ program on the library's planner."""
import os
import subprocess

import zkmetal_amd as zk

LIBDIR = os.path.dirname(zk.LIB_PATH)


def run_cpp(tmp_path, source):
    src, exe = tmp_path / "program.cpp", tmp_path / "program"
    src.write_text(source)
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I",
                        os.path.join(LIBDIR, "csrc"), str(src), "-o", str(exe), zk.LIB_PATH,
                        f"-Wl,-rpath,{LIBDIR}", "-L/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
