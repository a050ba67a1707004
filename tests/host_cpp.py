"""Small C++ programs that call the library's own host functions, on the CPU.

A program includes the source file whose functions it calls; kernels and other
files stay unresolved (nothing that it calls launches or allocates)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run(name, tmp_path):
    """compile tests/cpp/<name>.cpp and run it: its output"""
    exe = os.path.join(tmp_path, name)
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        f"-I{ROOT}/include", f"-I{ROOT}/oibvh_amd/csrc", f"{ROOT}/tests/cpp/{name}.cpp", "-o", exe,
                        "-Wl,--unresolved-symbols=ignore-all"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
