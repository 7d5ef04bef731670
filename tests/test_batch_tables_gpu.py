"""The argument tables of a batched sweep, which grow with members times
steps, are given back when a call ends, but for a few MB."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_tables_of_long_batches_are_given_back():
    import torch
    from rakali_amd import Grid
    from rakali_amd.adjoint import GaugeMisfit, backward_many, forward_many
    steps, n = 900, 8
    grids, sess = [], []
    for m in range(n):
        nx, ny = 16 + m, 12
        g = Grid(nx, ny, 10.0, 10.0, bc=("tidal", "wall", "wall", "wall"), manning_n=0.03, t_end=1e9, tidal_amplitude=0.1)
        g.set_field("b", np.full((nx, ny), -5.0, order="F"))
        g.set_field("h", np.full((nx, ny), 5.0, order="F"))
        g.use_manning_field(True)
        grids.append(g)
        sess.append(GaugeMisfit(g, steps, 30, gauges=[(3, 4)], targets=np.zeros((steps, 1))))
    free = []
    for _ in range(2):
        losses = forward_many(sess)
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        backward_many(sess)
        free.append((before, torch.cuda.mem_get_info()[0]))
    print(f"[batch tables] free before and after each sweep: {free}", flush=True)
    assert np.isfinite(losses).all()
    # 30 MB of tables a sweep; 4 MB may stay, and allocations are rounded to 2 MB
    assert all(before - after <= (6 << 20) for before, after in free)
    for s, g in zip(sess, grids):
        s.close()
        g.close()
