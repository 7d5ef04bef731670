"""The stage kernels' row path at the sizes and values where it can go wrong.

Strips own 60 columns between two halo columns, the last strip at least two;
tiles have 1 to 20 rows by the grid's size.  Rows without values of extreme
size are evaluated with selects, shared reciprocals and (for spacings of at
most 50 significant bits) two-operation quotients, the others with plain
divisions.  Every result must be the oracle's bits, and the bits of the same
run with every row on plain divisions."""
import struct

import numpy as np
import pytest


def _bits(x):
    return struct.unpack("<q", struct.pack("<d", x))[0]


def _double(i):
    return struct.unpack("<d", struct.pack("<q", i))[0]


def test_kp07_depth_is_the_first_depth_out_of_the_band():
    """h < KP07_DEPTH decides ((h h) h) h < DESING_EPS^4 for every h."""
    h, eps4 = float.fromhex("0x1.3a92a30553261p-13"), 5.062499999999998e-16
    below = _double(_bits(h) - 1)
    assert ((h * h) * h) * h >= eps4 and ((below * below) * below) * below < eps4


def _run(scn, steps, mode=0, tile_rows=0, **kw):
    from conftest import make_grid
    g = make_grid(scn, **kw)
    g.set_fast_path(mode)
    g.tile_rows = tile_rows
    g.step(steps)
    out = {k: g.get_field(k) for k in ("h", "hu", "hv")}, g.clock
    g.close()
    return out


def _check(scn, steps, tile_rows=0, **kw):
    from conftest import run_oracle
    got, clock = _run(scn, steps, 0, tile_rows, **kw)
    plain, clock2 = _run(scn, steps, -1, tile_rows, **kw)
    sim, ref = run_oracle(scn, steps, **kw)
    assert clock == clock2 and clock[0] == sim.t and clock[1] == sim.dt
    for k in ref:
        assert np.array_equal(got[k], ref[k]), k
        assert np.array_equal(plain[k], ref[k]), k


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny", [(2, 2), (2, 61), (59, 3), (60, 9), (61, 10), (62, 2), (119, 21), (121, 33),
                                   (181, 1), (181, 130), (301, 203)])
@pytest.mark.parametrize("bc", [("tidal", "wall", "open", "clamped"), ("chapman", "chapman", "chapman", "chapman")])
def test_strip_and_tile_remainders(nx, ny, bc):
    from rakali_amd import scenarios as S
    if ny == 1:
        nx, ny = ny + 1, nx   # two columns, many rows
    scn = S.wetdry_islands(nx=nx, ny=ny, steps=12, bc=bc)
    print(f"[strips] {nx}x{ny} {bc}", flush=True)
    _check(scn, 12, clamped_elevation=0.25)
    _check(scn, 6, tile_rows=1, clamped_elevation=0.25)


@pytest.mark.gpu
@pytest.mark.parametrize("dx,dy", [(10.0, 10.0), (62.5, 10.0), (0.1, 0.1), (10.1, 10.1), (7.3, 20.0), (1.0 / 3.0, 0.7)])
@pytest.mark.parametrize("hllc", [True, False])
def test_spacings(dx, dy, hllc):
    """Two-operation and shared-reciprocal quotients, one CFL maximum or two."""
    from rakali_amd import scenarios as S
    scn = S.wetdry_islands(nx=133, ny=47, steps=20, use_hllc=hllc)
    scn.dx, scn.dy = dx, dy
    print(f"[spacing] {dx} {dy} hllc={hllc}", flush=True)
    _check(scn, 20)


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["films", "tiny", "huge", "weak_friction", "strong_gravity"])
def test_values_at_the_row_paths_limits(case):
    """Depths at the dry tolerance and around the KP07 band, values below
    2^-300 and above 2^40, frictions and gravities outside the row path's
    ranges."""
    from rakali_amd import scenarios as S
    scn = S.wetdry_islands(nx=125, ny=40, steps=8)
    rng = np.random.default_rng(17)
    idx = rng.choice(scn.nx * scn.ny, 300, replace=False)
    kp = float.fromhex("0x1.3a92a30553261p-13")
    h, hu, hv, b = (np.array(a, order="F") for a in (scn.h, scn.hu, scn.hv, scn.b))
    kw = {}
    if case == "films":
        depths = np.array([1.0e-6, np.nextafter(1.0e-6, 0.0), np.nextafter(1.0e-6, 1.0), kp, _double(_bits(kp) - 1), 5e-5,
                           1.0e-3, np.nextafter(1.0e-3, 0.0)])
        h.reshape(-1, order="F")[idx] = rng.choice(depths, 300)
        hu.reshape(-1, order="F")[idx] = 1e-4 * rng.normal(size=300)
        hv.reshape(-1, order="F")[idx] = 1e-2 * rng.normal(size=300)   # some beyond the Froude backstop
    elif case == "tiny":
        hu.reshape(-1, order="F")[idx] = rng.choice([1e-305, -3e-310, 5e-320, 2.5e-91, -1e-90], 300)
        hv.reshape(-1, order="F")[idx[:100]] = 1e-320
        b.reshape(-1, order="F")[idx[:40]] = rng.choice([1e-310, -4e-320, 0.0], 40)
        h.reshape(-1, order="F")[idx[40:60]] = 1e-303
    elif case == "huge":
        h.reshape(-1, order="F")[idx[:5]] = [1.2e12, 3e12, 1e15, 1e20, 5e12]
        hu.reshape(-1, order="F")[idx[5:8]] = [1e14, -1e13, 2e12]
        b.reshape(-1, order="F")[idx[8:10]] = [-2e12, 3e12]
    elif case == "weak_friction":
        kw = dict(manning_n=1e-120)
    else:
        kw = dict(g=2.0e6)
    scn.h, scn.hu, scn.hv, scn.b = h, hu, hv, b
    print(f"[limits] {case}", flush=True)
    _check(scn, 8, **kw)
