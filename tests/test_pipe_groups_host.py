"""Group tables of the pipelined passes against a direct enumeration (CPU)."""

import ctypes
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = tmp_path_factory.mktemp("pipe") / "pipe_groups.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC",
                    str(ROOT / "tests/native/pipe_groups_check.cpp"),
                    str(ROOT / "ffsim_amd/csrc/host_core.cpp"), "-o", str(out)], check=True)
    return ctypes.CDLL(str(out))


# (window, electrons, 16-byte units per string)
CASES = [(6, 3, 8), (7, 2, 8), (12, 6, 8), (12, 4, 8), (13, 7, 4), (13, 6, 4), (14, 7, 2),
         (14, 5, 2), (15, 8, 1), (15, 7, 1), (16, 5, 1), (16, 1, 8), (16, 15, 8), (14, 14, 8),
         (10, 5, 16), (11, 6, 16), (6, 1, 16)]


@pytest.mark.parametrize("merge", [0, 1])
@pytest.mark.parametrize("w,kp,units", CASES)
def test_groups_and_schedule(lib, w, kp, units, merge):
    per_chunk = 64 // (units * (2 if merge else 1))
    assert lib.check_pipe_groups(w, kp, merge, units, per_chunk) == 0
