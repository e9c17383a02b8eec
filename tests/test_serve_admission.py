"""The job server's admission on a model of the context calls, no GPU: jobs
whose estimates fit the budget together run together, whatever the packed NW
kernels' scratch could take beside them, within the budget."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_jobs_that_fit_run_together(tmp_path):
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "serve_check.cpp"),
                    os.path.join(ROOT, "crispy_amd", "csrc", "serve.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.stdout.strip() == "ok", r.stdout + r.stderr
