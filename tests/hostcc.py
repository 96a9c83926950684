"""Compiles a C++ snippet against the library's host/device headers and runs
it on the CPU: the constants and rules that host code and kernels share."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run(tmp_path, body, include="internal.h"):
    src, exe = tmp_path / "snippet.cpp", tmp_path / "snippet"
    src.write_text('#include <cstdio>\n#include <cstdlib>\n#include "%s"\nusing namespace dm;\n'
                   "int main() {\n%s\nreturn 0;\n}\n" % (include, body))
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "dumato_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
