"""The rules by which the workgroups of a resident solve share memory
(csrc/rt_resident.h), run on the host under random interleavings
(tests/cpp/test_resident.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_shared_words_under_random_interleavings(tmp_path):
    exe = str(tmp_path / "test_resident")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "rheotool_amd", "csrc"), "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "test_resident.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK"), r.stdout + r.stderr
