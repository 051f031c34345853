"""Runs tests/cpp/test_stage_scratch.cpp: which scratch of the stage calls may be freed when
(no GPU)."""
import os
import subprocess

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "bin")


def test_cpp_stage_scratch():
    r = subprocess.run([os.path.join(BIN, "test_stage_scratch")], capture_output=True, text=True,
                       timeout=60)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    assert "All tests passed." in r.stdout
