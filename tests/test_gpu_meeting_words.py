"""A step after one whose bounded wait gave up: tests/cpp/meeting_words.cpp leaves the meeting words
of the sorts and the colouring as such a wait does, from the host, and runs a step's first launch and
a sort in several workgroups through the library."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "axiom-physics-engine_amd")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def build(tmp_path):
    exe = str(tmp_path / "meeting_words")
    cmd = ["g++", "-std=c++20", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
           "-I", os.path.join(ROOT, "include"), "-I", os.path.join(PKG, "csrc"),
           os.path.join(ROOT, "tests", "cpp", "meeting_words.cpp"), "-L", PKG, "-laxm",
           "-L", os.path.join(ROCM, "lib"), "-lamdhip64", "-Wl,-rpath," + PKG, "-Wl,-rpath," + os.path.join(ROCM, "lib"),
           "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


def test_builds(axm, tmp_path):
    build(tmp_path)


@pytest.mark.gpu
def test_step_starts_from_clear_meeting_words(axm, gpu, tmp_path):
    exe = build(tmp_path)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "OK", r.stdout + r.stderr
