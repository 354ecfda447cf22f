"""Builds and runs the C++ programs of tests/host_checks (host code of the engine
checked without a device; g++ only)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "lammps-mlip-package_amd", "csrc")


def run(folder, name, sources=(), args=()):
    """Compiles tests/host_checks/<name>.cpp with the named sources of csrc into
    `folder`, runs it and returns its output; a non-zero exit raises."""
    exe = os.path.join(str(folder), name)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-I", CSRC, "-o", exe,
                    os.path.join(HERE, "host_checks", name + ".cpp")] + [os.path.join(CSRC, s) for s in sources],
                   check=True)
    p = subprocess.run([exe] + [str(a) for a in args], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout[-4000:] + p.stderr[-4000:]
    return p.stdout
