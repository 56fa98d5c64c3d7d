"""A download's ring of chunks and its helper threads on the host: every value arrives, and no helper outlives what
started it (tests/cpp/ring_test.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_ring_and_helpers(tmp_path):
    exe = str(tmp_path / "ring_test")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-pthread",
                    os.path.join(HERE, "cpp", "ring_test.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "ok ring" in r.stdout, r.stdout + r.stderr
