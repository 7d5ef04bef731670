"""The face reverses at the sizes where their tiles can go wrong: strips of
60 and of 64 columns with remainders, rows that end inside a workgroup's, both
edges of a direction in one tile, each with every kind of edge; cell by cell
against the host reference adjoint."""
import numpy as np
import pytest

from test_adjoint_gpu import CFG, generic_state, gpu_grid, load

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ref(tmp_path_factory):
    import adjref
    return adjref.build(tmp_path_factory.mktemp("adjref"))


EDGES = [("tidal", "wall", "open", "tidal"), ("wall", "tidal", "tidal", "wall"),
         ("clamped", "inflow", "wall", "open"), ("open", "clamped", "discharge", "tidal")]


@pytest.mark.parametrize("nx, ny", [(2, 2), (2, 9), (3, 61), (59, 4), (60, 5), (61, 3), (62, 6), (64, 8), (65, 9), (119, 2),
                                    (121, 7), (129, 13)])
@pytest.mark.parametrize("bc", EDGES)
def test_face_reverses_at_tile_edges(ref, nx, ny, bc):
    import adjref
    from rakali_amd.adjoint import GaugeMisfit
    steps, hllc = 4, (nx + ny) % 2 == 0
    rng, b, n, h, hu, hv = generic_state(nx, ny, 7 * nx + ny)
    gauges = [(int(rng.integers(0, nx)), int(rng.integers(0, ny))) for _ in range(6)]
    tgt = rng.normal(0.0, 0.05, (steps, len(gauges)))
    cfg = dict(CFG, bc=bc, hllc=hllc, coriolis_f=0.0)
    loss_ref, want = adjref.run(ref, cfg, b, n, h, hu, hv, steps, gauges, tgt)
    print(f"[adjoint tiles] {nx}x{ny} {bc} hllc={hllc}", flush=True)
    g = gpu_grid(nx, ny, cfg, hllc, bc, 0.0)
    load(g, b, n, h, hu, hv)
    sess = GaugeMisfit(g, steps, 3, gauges, tgt)
    loss = sess.forward()
    sess.backward()
    assert abs(loss - loss_ref) <= 1e-12 * abs(loss_ref)
    for k in ("b", "n", "h", "hu", "hv"):
        got = sess.gradient(k)
        assert np.abs(got - want[k]).max() <= 1e-9 * np.abs(want[k]).max(), k
    sess.close()
    g.close()
