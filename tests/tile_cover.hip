// Host check of the stage tiles (set_tiles, tile_at, tile_range, tile_lane):
// the tiles of a launch own every cell exactly once, and what their lanes read
// lies in the plane.  Arguments: nx ny ty pack; prints the number of tiles.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "swe_kernels.hpp"

using namespace rk;

int main(int argc, char** argv) {
    for (int a = 1; a + 3 < argc; a += 4) {
        GridDesc d{};
        d.nx = atoi(argv[a]);
        d.ny = atoi(argv[a + 1]);
        d.pitch = (d.nx + 15) / 16 * 16;
        d.plane = d.pitch * d.ny;
        for (int e = 0; e < 4; ++e) d.bc[e] = e % 2 ? BC_WALL : BC_TIDAL;
        set_tiles(d, atoi(argv[a + 2]), atoi(argv[a + 3]) != 0);
        std::vector<int> owned((size_t)d.nx * d.ny, 0), slots((size_t)d.nstrips * d.nsegs, 0);
        for (int t = 0; t < d.ntiles; ++t) {
            const TileAt w = tile_at(d, t);
            int x0, x1, j0, j1;
            tile_range(d.nx, OWN, d.nstrips, w.strip, x0, x1);
            tile_range(d.ny, d.ty, d.nsegs, w.seg, j0, j1);
            for (int k = 0; k < w.count; ++k) slots[(size_t)(w.seg + k) * d.nstrips + w.strip] += 1;
            if (w.count > 1 && (j0 < HALO || j0 + w.count * d.ty + HALO > d.ny || j1 - j0 != d.ty)) return printf("ghost rows\n"), 1;
            for (int lane = 0; lane < WAVE; ++lane) {
                const bool edge = x0 < HALO || x0 + OWN + HALO > d.nx;
                const TileLane l = edge ? tile_lane<true>(d, w, x0, x1, lane) : tile_lane<false>(d, w, x0, x1, lane);
                const int lo = j0 < HALO ? 0 : j0 - HALO, hi = j1 + HALO > d.ny ? d.ny : j1 + HALO;
                if (l.at + lo * d.pitch < 0 || l.at + (hi - 1) * d.pitch >= d.plane) return printf("outside the plane\n"), 1;
                if (l.own && l.at != l.c + l.row * d.pitch) return printf("source of an own column\n"), 1;
                if (l.own)
                    for (int j = j0; j < j1; ++j) owned[(size_t)(j + l.row) * d.nx + l.c] += 1;
            }
        }
        for (int n : owned) if (n != 1) return printf("cells owned %d times\n", n), 1;
        for (int n : slots) if (n != 1) return printf("segments listed %d times\n", n), 1;
        printf("%d\n", d.ntiles);
    }
    return 0;
}
