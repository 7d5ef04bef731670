"""The stage tiles of a launch on the host (tests/tile_cover.hip, built here
with hipcc): every cell is owned once and every read lies in the plane, with and
without narrow last strips packed several segments to a wavefront."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def cover(tmp_path_factory):
    exe = tmp_path_factory.mktemp("tiles") / "tile_cover"
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    subprocess.run([hipcc, "-O1", "-std=c++17", "--offload-arch=gfx950", "-ffp-contract=off", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-I", str(ROOT / "rakali_amd" / "csrc"), "-I", str(ROOT / "include"),
                    str(ROOT / "tests" / "tile_cover.hip"), "-o", str(exe)], check=True)

    def run(cases):
        r = subprocess.run([str(exe), *(str(int(v)) for c in cases for v in c)], capture_output=True, text=True)
        out = r.stdout.split("\n")
        assert r.returncode == 0, (cases[len(out) - 2], out[-2:])
        return [int(v) for v in out if v]
    return run


def test_every_cell_is_owned_once(cover):
    cases = [(nx, ny, ty, pack) for nx in (*range(2, 94), 120, 121, 122, 128, 148, 149, 181, 256) for ny in (2, 3, 7, 40, 41)
             for ty in (1, 2, 3, 10, 20) for pack in (0, 1)]
    for k in range(0, len(cases), 1000):
        cover(cases[k:k + 1000])


def test_narrow_strips_share_wavefronts(cover):
    """64 columns are a full strip and one of 4, of which eight segments fit a
    wavefront; 89 columns leave 29, too many for two."""
    assert cover([(64, 1000, 10, 1)]) == [100 + 13 + 2] and cover([(89, 1000, 10, 1)]) == [200]
    assert cover([(64, 1000, 10, 0)]) == [200]
