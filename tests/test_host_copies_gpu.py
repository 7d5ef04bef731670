"""Uploads and downloads through pinned pieces: one piece, its exact size,
several, a row wider than a piece, wider leading dimensions, pinned arrays."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PIECE = (2 << 20) // 8   # values


def _roundtrip(grid_lib, up, down, nx, ny, ld, rng, alloc=np.empty):
    src = alloc((ny, ld))
    src[...] = rng.random((ny, ld))
    dst = alloc((ny, ld))
    dst[...] = -1.0
    assert up(src.ctypes.data_as(ctypes.c_void_p), ld) == 0
    assert down(dst.ctypes.data_as(ctypes.c_void_p), ld) == 0
    assert np.array_equal(dst[:, :nx], src[:, :nx])
    assert (dst[:, nx:] == -1.0).all()


@pytest.mark.parametrize("nx,ny", [(2, 2), (130, 97), (512, 512), (512, 513), (1000, 524), (1023, 1025), (PIECE, 2),
                                   (PIECE + 1, 2), (PIECE // 2 + 1, 5), (PIECE // 2, 4)])
def test_grid_planes(nx, ny):
    from rakali_amd import Grid
    from rakali_amd.grid import FIELDS
    print(f"[copies] {nx}x{ny}", flush=True)
    g = Grid(nx, ny, 1.0, 1.0, bc=("wall",) * 4)
    rng = np.random.default_rng(nx + ny)
    for ld in (nx, nx + 4):
        _roundtrip(g._lib, lambda p, d: g._lib.rkg_upload(g.handle, FIELDS["h"], p, d),
                   lambda p, d: g._lib.rkg_download(g.handle, FIELDS["h"], p, d), nx, ny, ld, rng)
    g.close()


def test_pinned_arrays():
    import torch
    from rakali_amd import Grid
    from rakali_amd.grid import FIELDS
    g = Grid(301, 203, 1.0, 1.0, bc=("wall",) * 4)
    _roundtrip(g._lib, lambda p, d: g._lib.rkg_upload(g.handle, FIELDS["hu"], p, d),
               lambda p, d: g._lib.rkg_download(g.handle, FIELDS["hu"], p, d), 301, 203, 305, np.random.default_rng(5),
               lambda shape: torch.empty(shape, dtype=torch.float64, pin_memory=True).numpy())
    g.close()


def test_ensemble_members_share_the_stage():
    from rakali_amd.ensemble import Ensemble
    sizes = [(16, 9), (700, 801), (64, 64), (1024, 256)]
    e = Ensemble([dict(nx=nx, ny=ny, dx=10.0, dy=10.0, bc=("wall",) * 4) for nx, ny in sizes])
    rng = np.random.default_rng(3)
    want = [np.asfortranarray(rng.random(s)) for s in sizes]
    for m, w in enumerate(want):
        e.set_field(m, "hv", w)
    for m, w in reversed(list(enumerate(want))):
        assert np.array_equal(e.get_field(m, "hv"), w)


def test_first_step_after_an_upload_is_not_captured():
    """Refused under capture, before anything is queued, and run as ever
    afterwards; a later step may be captured and replayed."""
    import torch
    from conftest import make_grid
    from rakali_amd import scenarios as S
    from rakali_amd._lib import RkgError
    scn = S.wetdry_islands(nx=75, ny=33, steps=4)
    want = make_grid(scn)
    want.step(4)
    s = torch.cuda.Stream()
    g = make_grid(scn, stream=s.cuda_stream)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=s):
        torch.zeros(1, device="cuda")
        with pytest.raises(RkgError):
            g.step(1)
    g.step(4)
    for k in ("h", "hu", "hv"):
        assert np.array_equal(g.get_field(k), want.get_field(k))
    assert g.clock == want.clock


@pytest.mark.parametrize("nx,ny", [(65536, 3), (65537, 3), (PIECE // 4, 2), (PIECE // 4 + 1, 2), (PIECE // 4 + 1, 3),
                                   (PIECE // 2, 2), (PIECE // 2 + 1, 3), (361, 363), (363, 362)])
def test_planes_at_the_limits_of_the_pieces(nx, ny):
    """Rows of just 512 KiB and planes of just 1 MiB, and one value more."""
    test_grid_planes(nx, ny)
