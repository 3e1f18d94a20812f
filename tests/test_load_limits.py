"""Limits of a circuit's load and store, on the CPU: which piece tables the
device checks and which fall back to the host (tests/native/piece_check.cpp),
transfers where no pinned memory can be had (tests/native/host_ring.cpp), and the
device memory of loads against the budget (tests/native/engine_memory.cpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# The programs define the HIP functions that they reach, so they are not linked
# with HIP; what the engine has beyond those stays unresolved.
@pytest.mark.parametrize("name,sources", [("piece_check", []), ("host_ring", []),
                                          ("engine_memory", ["ckt_engine.cpp", "ckt_generator.cpp"])])
def test_native(tmp_path, name, sources):
    exe, says = str(tmp_path / name), name.replace("_", " ") + ": ok"
    csrc = os.path.join(ROOT, "legionorigins_amd", "csrc")
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + csrc,
                        "-I" + os.path.join(ROOT, "include"), "-I/opt/rocm/include",
                        os.path.join(ROOT, "tests", "native", name + ".cpp"),
                        *[os.path.join(csrc, s) for s in sources], "-o", exe, "-lpthread",
                        "-Wl,--unresolved-symbols=ignore-all"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and says in r.stdout, r.stdout[-3000:] + r.stderr[-3000:]
