"""The library's host code on the CPU: every source compiled without its kernels, under the address sanitizer, and linked against a
stub of the HIP runtime (hip_stub.hpp) that records launches.  A test brings a program's main()."""
import os
import subprocess

from frink_amd import build as fb

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# (unoptimized: a read past a parameter is otherwise undefined before the sanitizer sees it)
FLAGS = ["-x", "hip", "--offload-arch=gfx950", "--offload-host-only", "-O0", "-g1", "-std=c++17", "-w", "-I", ROOT, "-Xarch_host", "-fsanitize=address"]


def build(directory, program):
    """The program's binary in `directory` (a pathlib.Path)."""
    (directory / "program.cpp").write_text('#include "tests/hip_stub.hpp"\n' + program)
    objs, procs = [], []
    for src in [str(directory / "program.cpp")] + [os.path.join(fb.CSRC, s) for s in fb.SOURCES]:
        objs.append(str(directory / (os.path.basename(src) + ".o")))
        procs.append(subprocess.Popen([fb.hipcc()] + FLAGS + ["-c", src, "-o", objs[-1]], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True))
    for p in procs:
        out, _ = p.communicate()
        assert p.returncode == 0, out[-3000:]
    binary = str(directory / "program")
    # (the kernels' images have no symbol in host-only objects)
    subprocess.check_call(["/opt/rocm/llvm/bin/clang++", "-fsanitize=address", "-no-pie", "-Wl,--unresolved-symbols=ignore-all"] + objs + ["-o", binary])
    return binary


def run(binary, text=""):
    """What the program prints; fails the test where it ends otherwise than well (the sanitizer's report included)."""
    r = subprocess.run([binary], input=text, capture_output=True, text=True, timeout=120, env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0, (r.stdout + r.stderr)[-3000:]
    return r.stdout
