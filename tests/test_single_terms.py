"""FP32 decisions of the one-wave kernel: the bounds of block records, on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_certain_decisions_agree_with_long_double(tmp_path):
    csrc = os.path.join(ROOT, "supertrack_amd", "csrc")
    exe = str(tmp_path / "single_terms_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "single_terms_check.cpp"), os.path.join(csrc, "layout.cpp"),
                    os.path.join(csrc, "parallel.cpp"), "-lpthread", "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    assert out.startswith("ok"), out
