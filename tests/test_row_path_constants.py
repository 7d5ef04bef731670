"""Constants of the row path as swe_core.hpp has them."""
import re
import struct
from pathlib import Path

CORE = Path(__file__).resolve().parents[1] / "rakali_amd" / "csrc" / "swe_core.hpp"


def _next(x, step):
    return struct.unpack("<d", struct.pack("<q", struct.unpack("<q", struct.pack("<d", x))[0] + step))[0]


def _h4(h):
    return ((h * h) * h) * h


def test_kp07_depth_of_the_header_is_the_first_out_of_the_band():
    """h < KP07_DEPTH stands for ((h h) h) h < eps4, DESING_EPS^4 as clamp_desing
    has it; the product is monotone in h, so the two neighbours decide."""
    text = CORE.read_text()
    depth = [float.fromhex(v) for v in re.findall(r"constexpr double KP07_DEPTH = (0x[0-9a-fp.+-]+);", text)]
    eps4 = {float(v) for v in re.findall(r"const double eps4 = ([0-9.e+-]+);", text)}
    assert len(depth) == 1 and len(eps4) == 1
    eps4 = eps4.pop()
    assert _h4(depth[0]) >= eps4 and _h4(_next(depth[0], -1)) < eps4
    assert re.search(r"constexpr double DESING_EPS = 1\.5e-4;", text) and abs(eps4 - 1.5e-4 ** 4) <= 1e-15 * eps4


def test_the_froude_margin_is_below_one():
    """num < h^2 (fr (1 - 2^-50)) decides num / h^2 <= fr with a relative room of
    2^-50 against three roundings."""
    assert re.search(r"fr_max_sq \* \(1\.0 - 0x1p-50\)", CORE.read_text())
    assert 1.0 - 2.0 ** -50 < 1.0 - 3 * 2.0 ** -53
