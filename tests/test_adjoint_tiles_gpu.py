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


@pytest.mark.parametrize("hllc", [True, False])
@pytest.mark.parametrize("rows", [0, 5])
def test_batched_forward_runs_equal_single_runs(hllc, rows):
    """One launch for all members: uneven sizes down to two cells, a member
    without gauges, an odd start parity, a second batch of another size."""
    from rakali_amd.adjoint import GaugeMisfit, backward_many, forward_many
    sizes, steps, K = [(2, 2), (61, 33), (130, 70), (200, 9), (3, 40)], 7, 3
    grids, sess, states = [], [], []
    for m, (nx, ny) in enumerate(sizes):
        rng, b, n, h, hu, hv = generic_state(nx, ny, 90 + m)
        g = gpu_grid(nx, ny, dict(CFG, dt=0.0), hllc, EDGES[m % 4], 1e-3 * (m % 2))
        g.tile_rows = rows
        k = 0 if m == 3 else 6
        gauges = [(int(rng.integers(0, nx)), int(rng.integers(0, ny))) for _ in range(k)]
        sess.append(GaugeMisfit(g, steps, K, gauges, rng.normal(0.0, 0.05, (steps, k))))
        grids.append(g)
        states.append((b, n, h, hu, hv))

    def start(m):
        load(grids[m], *states[m])
        if m == 1:
            grids[m].step(1)

    def result(m):
        return ({k: grids[m].get_field(k) for k in ("h", "hu", "hv")}, grids[m].clock, sess[m].gauge_eta(),
                {k: sess[m].gradient(k) for k in ("b", "n", "h")})

    for batch in ([0, 1, 2, 3, 4], [4, 2], [3, 0, 1, 2]):
        print(f"[batched forward] {batch} hllc={hllc} rows={rows}", flush=True)
        for m in batch:
            start(m)
        losses = forward_many([sess[m] for m in batch])
        backward_many([sess[m] for m in batch])
        many = [result(m) for m in batch]
        for i, m in enumerate(batch):
            start(m)
            assert sess[m].forward() == losses[i]
            sess[m].backward()
            f, clock, eta, grad = result(m)
            assert clock == many[i][1] and np.array_equal(eta, many[i][2])
            assert all(np.array_equal(f[k], many[i][0][k]) for k in f)
            assert all(np.array_equal(grad[k], many[i][3][k]) for k in grad)
    for s in sess:
        s.close()
    for g in grids:
        g.close()
