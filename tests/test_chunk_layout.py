"""The group chunks of pipelined answers: tests/cpp/test_chunks.cpp over
chunks.h, for every divisor of up to 2304 groups, with and without the
split of the first and last chunk, chunks that end with a response
ciphertext and chunks that straddle two."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_chain_runs_on_one_stream(tmp_path):
    exe = str(tmp_path / "test_chunks")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "inspire-gpu_amd", "csrc", "server"),
                    os.path.join(ROOT, "tests", "cpp", "test_chunks.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
    assert "layouts checked" in r.stdout
