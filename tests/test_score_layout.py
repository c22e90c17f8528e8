"""Alignment and extent of the score kernel's LDS for every number of taps, by
the host compiler."""
import subprocess
from pathlib import Path

HOST = Path(__file__).resolve().parent / "host"
CSRC = HOST.parents[1] / "ctas_amd" / "csrc"


def test_score_layout(tmp_path):
    exe = tmp_path / "score_layout_test"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", str(CSRC), str(HOST / "score_layout_test.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
