"""The one-wave kernel's track flags on the CPU (tests/wave_flags_check.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_wave_flags_bound_what_a_flush_keeps(tmp_path):
    exe = str(tmp_path / "wave_flags_check")
    csrc = os.path.join(ROOT, "supertrack_amd", "csrc")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "wave_flags_check.cpp"), os.path.join(csrc, "layout.cpp"),
                    os.path.join(csrc, "parallel.cpp"), "-lpthread", "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and "ALL OK" in out.stdout, out.stdout + out.stderr
