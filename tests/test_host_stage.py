"""The crew that stages host queries: tests/cpp/test_host_stage.cpp over
host_stage.h, also where its threads cannot all be made."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_jobs_with_every_number_of_helpers(tmp_path):
    exe = str(tmp_path / "test_host_stage")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I",
                    os.path.join(ROOT, "inspire-gpu_amd", "csrc", "server"),
                    os.path.join(ROOT, "tests", "cpp", "test_host_stage.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
    assert "host stage checks passed" in r.stdout
