"""The pools behind host-array calls and per-call scratch (pools.cpp), built by
the host compiler on a stand-in for HIP (tests/host)."""
import subprocess
from pathlib import Path

import pytest

HOST = Path(__file__).resolve().parent / "host"
CSRC = HOST.parents[1] / "ctas_amd" / "csrc"


@pytest.fixture(scope="session")
def pools_test(tmp_path_factory):
    exe = tmp_path_factory.mktemp("pools") / "pools_test"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", str(HOST), "-I", str(CSRC), str(HOST / "pools_test.cpp"),
                    str(CSRC / "pools.cpp"), "-o", str(exe), "-pthread"], check=True)
    return exe


@pytest.mark.parametrize("case", ["copies", "device", "streams", "refused", "end"])
def test_pools(pools_test, case):
    r = subprocess.run([str(pools_test), case], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
