"""Compiles a C++ snippet against the library's host/device headers and runs
it on the CPU: the constants and rules that host code and kernels share; with
link, against the built library too."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIBDIR = os.path.join(ROOT, "dumato_amd")
LIB = ["-L" + LIBDIR, "-ldumato_amd", "-Wl,-rpath," + LIBDIR, "-L/opt/rocm/lib", "-lamdhip64",
       "-Wl,-rpath,/opt/rocm/lib"]


def run(tmp_path, body, include="internal.h", link=False):
    src, exe = tmp_path / "snippet.cpp", tmp_path / "snippet"
    src.write_text('#include <cstdio>\n#include <cstdlib>\n#include "%s"\nusing namespace dm;\n'
                   "int main() {\n%s\nreturn 0;\n}\n" % (include, body))
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "dumato_amd", "csrc"),
                    str(src), "-o", str(exe)] + (LIB if link else []), check=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
