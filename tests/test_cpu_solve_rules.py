"""Dispatch rules of the solver's sweeps that the device evaluates, compiled for the host
(tests/cpp/solve_rules.cpp) and checked at their edges."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "axiom-physics-engine_amd")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def test_register_sweep_rule(tmp_path):
    exe = str(tmp_path / "solve_rules")
    cmd = ["g++", "-std=c++20", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
           "-I", os.path.join(ROOT, "include"), "-I", os.path.join(PKG, "csrc"),
           os.path.join(ROOT, "tests", "cpp", "solve_rules.cpp"), "-L", os.path.join(ROCM, "lib"), "-lamdhip64",
           "-Wl,-rpath," + os.path.join(ROCM, "lib"), "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "OK", r.stdout + r.stderr
