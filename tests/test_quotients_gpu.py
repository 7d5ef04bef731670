"""The shared reciprocal's quotients are the device's division on the operands where
a reciprocal off by one neighbour could show (tests/quotients.hip, built here
with hipcc; the enumeration and its reason are there)."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def _run(tmp_path):
    exe = tmp_path / "quotients"
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    subprocess.run([hipcc, "-O2", "-std=c++17", "--offload-arch=gfx950", "-ffp-contract=off", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-I", str(ROOT / "rakali_amd" / "csrc"), "-I", str(ROOT / "include"),
                    str(ROOT / "tests" / "quotients.hip"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    print(r.stdout, flush=True)
    assert r.returncode == 0
    return r.stdout


def test_the_pairs_tell_a_wrong_reciprocal(tmp_path):
    out = _run(tmp_path)
    n, pairs, wrong = map(int, re.search(r"denominators (\d+) pairs (\d+) wrong_with_the_other_neighbour (\d+)", out).groups())
    assert "nearest reciprocal wrong" not in out
    assert n > 0 and pairs > 0 and wrong > pairs // 10


@pytest.mark.gpu
def test_device_quotients_are_the_divisions(tmp_path):
    wrong = re.findall(r"device exponent (-?\d+) wrong (\d+)", _run(tmp_path))
    assert len(wrong) == 5 and all(int(w) == 0 for _, w in wrong), wrong
