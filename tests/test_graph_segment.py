"""The captured launch sequences' bookkeeping on a model of the HIP runtime, no
GPU: what runs is what was asked for, no graph is built for runs that do not
come again, and an instantiated graph is only updated with arguments of its own
kernels, and only updated or destroyed when its last launch has ended."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def test_run_segment(tmp_path):
    if not os.path.isdir(os.path.join(ROCM, "include", "hip")):
        pytest.skip("no HIP headers")
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "crispy_amd", "csrc"),
                    os.path.join(ROOT, "tests", "graph_segment_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.stdout.strip() == "ok", r.stdout + r.stderr
