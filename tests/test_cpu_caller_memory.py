"""Device vectors are used in place only where they lie whole on the solver's GPU: host memory, another GPU's and
vectors longer than their allocation keep the copies (tests/cpp/caller_memory_check.cpp on the rule of
ins-solver_amd/csrc/caller_memory.h)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_memory_taken_in_place(tmp_path):
    exe = str(tmp_path / "caller_memory_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "ins-solver_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "caller_memory_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
