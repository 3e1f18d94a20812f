"""Limits of a circuit's load, on the CPU: which piece tables the device checks
and which fall back to the host (tests/native/piece_check.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_piece_tables_fit_their_launch(tmp_path):
    from legionorigins_amd import build as B
    exe = str(tmp_path / "piece_check")
    r = subprocess.run([B.hipcc(), "-O1", "-std=c++17", "--offload-arch=gfx950", "-x", "hip",
                        "-I" + os.path.join(ROOT, "legionorigins_amd", "csrc"),
                        os.path.join(ROOT, "tests", "native", "piece_check.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "piece check: ok" in r.stdout, r.stdout[-3000:]
