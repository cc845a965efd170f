"""The fused CG's device state: no wave of a launch reads what another wave of it writes, and launches after
the end change nothing and stay a small part of the run (tests/cpp/pcg_state_check.cpp on the functions of ins-solver_amd/csrc/pcg_state.h
that the kernels call)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_state_accesses(tmp_path):
    exe = str(tmp_path / "pcg_state_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "ins-solver_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "pcg_state_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout[-3000:]
