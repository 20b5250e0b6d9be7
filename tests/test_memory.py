"""The library's memory code on the CPU: bsx_mem.hip built with g++ over a
stand-in for the HIP allocator (tests/memory), and that no other source
allocates past it."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "bsoft_amd", "csrc")


def test_workspaces_and_their_return(tmp_path):
    """Kept buffers are reused and bounded, are given back where any allocation
    of the library would fail and on request, and are never in two hands."""
    exe = tmp_path / "memory_check"
    here = os.path.join(ROOT, "tests", "memory")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-I", here, "-I", CSRC,
                    "-x", "c++", os.path.join(here, "memory_check.cpp"), os.path.join(CSRC, "bsx_mem.hip"),
                    "-pthread", "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr


def test_every_allocation_goes_through_it():
    """No source but bsx_mem.hip calls the runtime's allocators."""
    for name in sorted(os.listdir(CSRC)):
        if name.endswith((".hip", ".h")) and name != "bsx_mem.hip":
            src = open(os.path.join(CSRC, name)).read()
            assert not re.search(r"\bhip(Host|Ext|Managed)?Malloc\w*\s*\(", src), name
