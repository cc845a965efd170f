"""The partial sums that the device kernels leave fit the buffers kept for them (tests/cpp/partials_check.cpp
on the counts of ins-solver_amd/csrc/partials.h, which the launches use)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_partials_fit_their_buffers(tmp_path):
    exe = str(tmp_path / "partials_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-I" + os.path.join(ROOT, "ins-solver_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "partials_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
