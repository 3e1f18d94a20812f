"""Limits of a circuit's load and store, on the CPU: which piece tables the
device checks and which fall back to the host (tests/native/piece_check.cpp),
and transfers where no pinned memory can be had (tests/native/host_ring.cpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# host_ring defines the HIP functions it calls, so it is not linked with HIP
@pytest.mark.parametrize("name,says", [("piece_check", "piece check: ok"),
                                       ("host_ring", "host ring: ok")])
def test_native(tmp_path, name, says):
    exe = str(tmp_path / name)
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__",
                        "-I" + os.path.join(ROOT, "legionorigins_amd", "csrc"),
                        "-I" + os.path.join(ROOT, "include"), "-I/opt/rocm/include",
                        os.path.join(ROOT, "tests", "native", name + ".cpp"), "-o", exe, "-lpthread"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and says in r.stdout, r.stdout[-3000:] + r.stderr[-3000:]
