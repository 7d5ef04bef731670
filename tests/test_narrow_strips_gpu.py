"""Grids whose last strip is narrow (28 columns or fewer): above 1024 tiles
several of its segments share a wavefront.  The packed launches give the
oracle's bits, and the bits of launches of few tall tiles, which are not
packed."""
import numpy as np
import pytest

from conftest import make_grid, run_oracle

pytestmark = pytest.mark.gpu

BC = {"ghosts": ("tidal", "wall", "open", "clamped"), "outflow": ("inflow", "tidal", "wall", "wall"),
      "chapman": ("chapman", "chapman", "open", "chapman")}


def _scn(nx, ny, bc, hllc=True):
    from rakali_amd import scenarios as S
    return S.wetdry_islands(nx=nx, ny=ny, steps=6, bc=BC[bc], use_hllc=hllc)


@pytest.mark.parametrize("nx,ny,rows", [(2, 1203, 1), (2, 1101, 1), (28, 1030, 1), (29, 1030, 1), (61, 700, 1), (62, 1030, 2),
                                        (64, 1801, 3), (75, 611, 1), (88, 523, 1), (121, 400, 1), (128, 1043, 3)])
@pytest.mark.parametrize("bc", list(BC))
def test_packed_segments_give_the_oracles_bits(nx, ny, rows, bc):
    scn = _scn(nx, ny, bc, hllc=nx % 2 == 0)
    print(f"[narrow] {nx}x{ny} rows={rows} {bc}", flush=True)
    over = dict(clamped_elevation=0.25, inflow_velocity=0.3)
    g = make_grid(scn, **over)
    g.tile_rows = rows
    g.step(6)
    got, clock = {k: g.get_field(k) for k in ("h", "hu", "hv")}, g.clock
    g.close()
    sim, ref = run_oracle(scn, 6, **over)
    assert clock[0] == sim.t and clock[1] == sim.dt
    for k in ref:
        assert np.array_equal(got[k], ref[k]), k


@pytest.mark.parametrize("scheme", ["rk2", "euler", "rk3", "rk43"])
@pytest.mark.parametrize("nx", [2, 64, 81])
@pytest.mark.parametrize("terms", ["plain", "all"])
def test_packed_source_terms_equal_unpacked(scheme, nx, terms):
    """Manning field, forcing, sponge, mass budget and the U^n copy."""
    ny = 1101
    scn = _scn(nx, ny, "ghosts")
    if terms == "all":
        scn.grid_kw["bc"] = ("tidal", "sponge", "sponge", "chapman")
    print(f"[narrow terms] {nx}x{ny} {scheme} {terms}", flush=True)
    out = []
    for rows in (1, 64):
        rng = np.random.default_rng(5)
        g = make_grid(scn, time_scheme=scheme, clamped_elevation=0.25)
        g.tile_rows = rows
        g.use_manning_field(True)
        g.set_field("n", np.asfortranarray(rng.uniform(0.0, 0.05, (nx, ny))))
        g.track_mass_budget(True)
        g.keep_rk_save(True)
        if terms == "all":
            g.forcing = True
            for k, a in (("wind_x", 0.1), ("wind_y", -0.1), ("atm_pressure", 40.0), ("precipitation", 1e-4)):
                g.set_field(k, np.asfortranarray(a * rng.uniform(0.0, 1.0, (nx, ny))))
            g.sponge = (9, 0.05, 1.0)
        g.step(5)
        out.append(({k: g.get_field(k) for k in ("h", "hu", "hv", "h0", "hu0", "hv0")}, g.clock, g.mass_out, g.mass_src,
                    g.total_mass()))
        g.close()
    a, b = out
    assert a[1] == b[1]
    for k in a[0]:
        assert np.array_equal(a[0][k], b[0][k]), k
    # sums over tiles in another order: 1e-12 of the mass, as the other budget tests
    assert abs(a[2] - b[2]) <= 1e-12 * a[4] and abs(a[3] - b[3]) <= 1e-12 * a[4]


@pytest.mark.parametrize("schedule", ["flat", "persistent"])
def test_packed_ensemble_members_equal_single_grids(schedule):
    from rakali_amd.ensemble import from_scenarios
    scns = [_scn(nx, ny, bc) for nx, ny in ((64, 300), (2, 257), (128, 200), (61, 9), (90, 211), (240, 150))
            for bc in ("ghosts", "outflow")]
    for s in scns:
        s.grid_kw.update(clamped_elevation=0.25, inflow_velocity=0.3)
    with from_scenarios(scns) as e:
        e.set_schedule(schedule, tile_rows=4)
        assert e.tiles < sum(-(-s.nx // 60) * -(-s.ny // 4) for s in scns)
        e.step(7)
        for m, s in enumerate(scns):
            g = make_grid(s)
            g.step(7)
            assert e.clock(m) == g.clock
            for k in ("h", "hu", "hv"):
                assert np.array_equal(e.get_field(m, k), g.get_field(k)), (m, k)
            g.close()


@pytest.mark.parametrize("many", [False, True])
def test_packed_replays_give_the_same_gradients(many):
    from rakali_amd.adjoint import GaugeMisfit, backward_many, forward_many
    res = []
    for rows in (1, 64):
        grids, sess = [], []
        for nx, ny in ((64, 1101), (2, 1101), (75, 40), (61, 211)):   # four: one run for all where they are many
            scn = _scn(nx, ny, "ghosts")
            g = make_grid(scn, clamped_elevation=0.25)
            g.tile_rows = rows
            g.use_manning_field(True)
            g.set_field("n", np.full((nx, ny), 0.03, order="F"))
            grids.append(g)
            sess.append(GaugeMisfit(g, 5, 3, gauges=[(0, 7), (1, ny // 2), (nx - 1, ny - 9)], targets=np.zeros((5, 3))))
        if many:
            loss = list(forward_many(sess))
            backward_many(sess)
        else:
            loss = [s.forward() for s in sess]
            for s in sess:
                s.backward()
        res.append((loss, [s.gradient(k) for s in sess for k in ("b", "n", "h", "hu", "hv")]))
        for s, g in zip(sess, grids):
            s.close()
            g.close()
    assert res[0][0] == res[1][0]
    for a, b in zip(res[0][1], res[1][1]):
        assert np.array_equal(a, b)
