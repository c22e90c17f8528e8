"""Which launches a batch of slices takes: groups of one centre, small tiles, and
none of them where the caller set a tile kind or a pass length. By the host
compiler."""
import subprocess
from pathlib import Path

HOST = Path(__file__).resolve().parent / "host"
CSRC = HOST.parents[1] / "ctas_amd" / "csrc"


def test_bp_plan(tmp_path):
    exe = tmp_path / "bp_plan_test"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", str(CSRC), str(HOST / "bp_plan_test.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[:2000]
