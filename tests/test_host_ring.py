"""The ring of pinned slots (stzpp_amd/csrc/host_copy.hpp) on the CPU:
tests/abi/host_ring.cpp compiles it with stand-ins for the HIP calls and lets
the memory for its threads run out after 0 to 8 allocations.  A copy arrives
whole all the same, by the threads that were started and the caller, and no
exception leaves the call."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_copies_without_memory_for_threads(tmp_path):
    exe = str(tmp_path / "host_ring")
    subprocess.run(["g++", "-O2", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "abi", "host_ring.cpp"), "-o", exe, "-lpthread"], check=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0 and p.stdout.strip() == "OK", p.stdout + p.stderr
