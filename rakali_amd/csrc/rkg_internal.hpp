// rkg_internal.hpp -- error reporting shared by the translation units of
// librakali_amd.so (not part of the ABI).
#pragma once

#include <hip/hip_runtime.h>

#include <cstring>
#include <mutex>

#include "../../include/rakali_amd.h"
#include "swe_kernels.hpp"

namespace rk {

// Records the message returned by rkg_last_error() on this thread.
__attribute__((visibility("hidden"), format(printf, 1, 2))) void set_error(const char* fmt, ...);

}  // namespace rk

namespace rk {
struct GaugeState;   // gauge stations and their time series (rkg_gauges.hip)

// Pinned memory between the planes of one grid or ensemble and its caller's
// pageable arrays.  A pitched copy to pageable memory goes row by row, 7 us
// each (768 x 700: 4.9 ms down, 6.5 ms up); to pinned memory it is one
// transfer at the link's rate (83 us) plus a copy in host memory (55 us).  A
// plane goes through in pieces, one in transfer while the host copies the
// other.  Uploads of wide rows go directly: the runtime takes a row of pageable
// memory faster than the host copies it (us, directly / through the stage: rows
// of 160 KB x 32 380 / 209, 320 KB x 4 68 / 76, 800 KB x 32 757 / 956; downloads
// of 800 KB x 32 1507 / 983).  Made on first use, at most 2 * PIECE bytes, freed
// with its owner; calls from several threads take turns.
struct HostStage {
    static constexpr size_t PIECE = (size_t)2 << 20, WIDEST_UP = (size_t)1 << 19;
    std::mutex lock;
    double* mem = nullptr;
    size_t bytes = 0;     // of mem
    ~HostStage();
};

// ny rows of nx values between a plane (rows `pitch` apart) and host memory
// (rows ld apart), complete on return.
__attribute__((visibility("hidden"))) hipError_t plane_to_host(HostStage& st, double* dst, size_t ld, const double* plane,
                                                               size_t pitch, size_t nx, size_t ny, hipStream_t stream);
__attribute__((visibility("hidden"))) hipError_t plane_from_host(HostStage& st, double* plane, size_t pitch, const double* src,
                                                                 size_t ld, size_t nx, size_t ny, hipStream_t stream);
}

// One grid: device buffers, stream and control slots (rkg_grid of the ABI).
struct rkg_grid {
    unsigned magic;
    rkg_config cfg;
    int device;
    hipStream_t stream;
    bool own_stream;     // the stream was made by rkg_create (this grid holds a reference to it)
    int refs;            // 1 for the caller's handle + 1 per attached adjoint session
    long long pitch;
    size_t plane;        // elements per field plane
    double* buf;         // 7 planes: A(h,hu,hv) B(h,hu,hv) bed
    double* save;        // 3 planes: U^n of the last step (RK save), or null
    double* nfield;      // per-cell Manning n (1 plane), or null
    double* cbuf;        // 3 planes: third stage buffer of rk3 / rk43, or null
    double* mpart;       // per-tile sums of both stages (mass budget): flux_h, then the sponge's
                         // change of h (2 x mpart_cap each), or null
    long long mpart_cap; // tiles per stage that mpart holds
    int scheme;          // RKG_TIME_*
    double* frc;         // 6 planes: wind stress x, y, atmospheric pressure, precipitation, and
                         // the pressure gradient x, y (from the pressure plane), or null
    bool forcing;        // forcing%active: the stage kernels apply the planes in frc
    bool frc_grad_stale; // the pressure plane may have changed since the gradient was taken
    bool frc_pres_out;   // a device pointer to the pressure plane was handed out
    int sponge_width;    // sponge relaxation next to RKG_BC_SPONGE edges (bc_params_t)
    double sponge_strength, sponge_h_ref;
    rk::CtrlSlot* ctrl;      // device [2]
    rk::CtrlSlot* ctrl_host; // pinned [2]
    double* mass_buf;    // device [MASS_BLOCKS + 2]: partial sums, total mass, precipitation sum
    double* mass_host;   // pinned [1]
    int parity;
    int ty;              // rows per stage tile, 0 = chosen from the grid size
    int fast_mode;       // rkg_set_fast_path: -1 runs every row with plain divisions
    bool speed_stale;
    bool prof;             // time each stage launch with events
    hipEvent_t ev[3];
    double prof_ms[2];     // accumulated stage-1 / stage-2 kernel time
    long long prof_n;
    rk::GaugeState* gauges;  // stations, or null
    rk::HostStage* stage;    // uploads and downloads from and to pageable memory
};

namespace rk {

constexpr unsigned GRID_MAGIC_LIVE = 0x72616B47u;  // 'rakG', rkg_grid::magic of a live grid
inline bool grid_valid(const rkg_grid* g) { return g != nullptr && g->magic == GRID_MAGIC_LIVE; }

// Holds / drops a reference to the grid's device state: an adjoint session
// retains its grid, so destroying the grid first leaves the session's
// buffers valid until the session is destroyed too (the grid is freed with
// its last reference).
void grid_retain(rkg_grid* g);
void grid_release(rkg_grid* g);

// The checks rkg_create applies to a configuration (sizes, spacing, tags);
// RKG_OK or an error code with the message set.
int validate_config(const rkg_config* c);

// RKG_ERR_HIP (with the message set) while `stream` is being captured: the
// speed maximum of an uploaded state is taken once, when the host sees the
// upload, and would otherwise be left to the captured graph's launch.
int refuse_capture(hipStream_t stream);

inline double* plane_ptr(rkg_grid* g, int k) { return g->buf + (size_t)k * g->plane; }

// Gauge recording around the step launches (rkg_gauges.hip): the steps one
// launch may take before the device series must be drained, the drain, the
// record after a step (slot p holds the state after it), and the release.
// Station (x, y) in metres: false when it lies outside the domain
// (compute_local_gauges, rki_gauges.F90:208-243); else its lower-left
// interpolation cell (c0, j0, 0-based interior) and weights
// (compute_interp_weights, :245-336).
bool station_weights(const rkg_config& c, double x, double y, int* c0, int* j0, double* wx, double* wy);

long long gauges_room(const rkg_grid* g);
int gauges_drain(rkg_grid* g);
// The record after a step together with its mass budget (if it has one);
// false when no gauges are recorded and nothing was launched.
bool gauges_after_step(rkg_grid* g, int p, const BudgetArgs& budget);
void gauges_free(rkg_grid* g);

inline double* field_ptr(rkg_grid* g, int field) {
    switch (field) {
    case RKG_FIELD_H: return plane_ptr(g, 0);
    case RKG_FIELD_HU: return plane_ptr(g, 1);
    case RKG_FIELD_HV: return plane_ptr(g, 2);
    case RKG_FIELD_B: return plane_ptr(g, 6);
    case RKG_FIELD_H0: return g->save ? g->save : nullptr;
    case RKG_FIELD_HU0: return g->save ? g->save + g->plane : nullptr;
    case RKG_FIELD_HV0: return g->save ? g->save + 2 * g->plane : nullptr;
    case RKG_FIELD_HS: return plane_ptr(g, 3);
    case RKG_FIELD_HUS: return plane_ptr(g, 4);
    case RKG_FIELD_HVS: return plane_ptr(g, 5);
    case RKG_FIELD_N: return g->nfield;
    case RKG_FIELD_WIND_X: return g->frc;
    case RKG_FIELD_WIND_Y: return g->frc ? g->frc + g->plane : nullptr;
    case RKG_FIELD_PRESSURE: return g->frc ? g->frc + 2 * g->plane : nullptr;
    case RKG_FIELD_PRECIP: return g->frc ? g->frc + 3 * g->plane : nullptr;
    case RKG_FIELD_BC_H:
    case RKG_FIELD_BC_HU:
    case RKG_FIELD_BC_HV:
    case RKG_FIELD_BC_PREV_H: {
        // the last step's last boundary call: its state and the previous
        // call's (rki_solver.F90:760-815 for SSP-RK2, :861-925 for the
        // generic stage loop); stage buffers B = planes 3-5, C = cbuf
        double* B = plane_ptr(g, 3);
        double* cur = nullptr;
        double* prev = nullptr;
        switch (g->scheme) {
        case RKG_TIME_EULER: cur = g->save; prev = g->save; break;   // U^n, after the pre-dt call on U^n
        case RKG_TIME_RK3: cur = g->cbuf; prev = B; break;           // stage 3 input, stage 2 input
        case RKG_TIME_RK43: cur = B; prev = g->cbuf; break;          // stage 4 input, stage 3 input
        default: cur = B; prev = g->save; break;                     // U*, U^n
        }
        if (!cur || !prev) return nullptr;
        if (field == RKG_FIELD_BC_PREV_H) return prev;
        return cur + (size_t)(field - RKG_FIELD_BC_H) * g->plane;
    }
    default: return nullptr;
    }
}

// Rows per stage tile; tiles(rows) counts a launch's tiles.  A tile costs half
// a row more than its rows (the march starts a row early), and a launch whose
// tiles are all resident lasts as long as one tile.  So a launch takes the
// shortest tiles, up to 3 rows, that still fit the chip's 3072 wavefront slots
// at once; else the shortest, up to 10, that leave two wavefronts on each of
// the 1024 SIMDs, which is enough to keep them busy and costs grids that run
// beside others less.  Larger launches run several tiles per slot: 10 rows,
// and 20 once there are 8192 tiles of 16, where the uneven end of a launch no
// longer matters.  Measured (us per step, one grid / each of three grids on
// their own streams):
//   200x100    1 row  23 / 9,    3 rows  32 / 13,   6 rows 49 / 19
//   400x300    1 row  31 / 15,   3 rows  33 / 15,   6 rows 49 / 21
//   512x512    2 rows 42 / 23,   1 row   48 / 31,   5 rows 46 / 23
//   701x515    3 rows 48 / 27,   7 rows  58 / 28,  10 rows 73 / 33
//   800x800    6 rows 70 / 40,   3 rows  71 / 45,  10 rows 92 / 43
//   1024x1024  10 rows 101 / 60, 5 rows  98 / 62,  20 rows 130 / 71
//   3000x2000  10 rows 370 / 345, 16 rows 403 / 338
//   4096x4096  20 rows 970 / 914, 10 rows 983 / 950, 32 rows 987 / 908
// and for ensembles (their tiles have 4 rows at least; nx and ny log-uniform):
//   4 of 64..200      4 rows 39, 8 rows 60, 32 rows 190
//   12 of 200..400    10 rows 127, 4 rows 111, 32 rows 203
//   16 of 128..768    10 rows 196, 20 rows 230, 32 rows 272
//   64 of 256x256     10 rows 279, 4 rows 291, 32 rows 350
//   32 of 512..1024   20 rows 1154, 10 rows 1175, 32 rows 1174
//   64 of 128..2048   20 rows 1926, 10 rows 1979, 32 rows 1931
template <class TILES>
int rows_for(TILES tiles, int least) {
    for (int rows = least; rows <= 3; ++rows)
        if (tiles(rows) <= 3 * 1024) return rows;
    for (int rows = least; rows <= 10; ++rows)
        if (tiles(rows) <= 2 * 1024) return rows;
    return tiles(16) >= 8192 ? 20 : 10;
}

inline long long grid_tiles(int nx, int ny, int rows) {
    return (long long)((nx + OWN - 1) / OWN) * ((ny + rows - 1) / rows);
}

// Whether a launch packs the segments of its narrow last strips (tile_at):
// `tiles` wavefronts without, `packed` with.  It pays where the launch is more
// than the chip's 3072 slots, or where it leaves the fullest of the 1024 SIMDs a
// wavefront less to run; with as many there a shared wavefront, which reads
// `pack` rows at a time, is the slower one.  us per step, unpacked / packed:
//   64x262144 1821 / 1104,  128x131072 1286 / 1038,  256x8192  180 / 164,
//   128x8192   123 / 104,   64x3000      47 / 39,    2x100000  383 / 82;
//   as many on a SIMD: 128x2048 41 / 45, 500x1000 51 / 55, 256x1024 41 / 43;
//   ensembles of 64 x 256^2 302 / 275, 256 x 128^2 358 / 302, 256 x 64^2 185 / 134
inline bool pack_pays(long long tiles, long long packed) {
    auto fullest = [](long long n) { return (n + 1023) / 1024; };
    return tiles > 3 * 1024 || fullest(packed) < fullest(tiles);
}

// The tiles of the n members of a launch.
inline void set_launch_tiles(GridDesc* d, int n, const int* ty) {
    long long tiles = 0, packed = 0;
    for (int m = 0; m < n; ++m) {
        set_tiles(d[m], ty[m], true);
        tiles += (long long)d[m].nstrips * d[m].nsegs;
        packed += d[m].ntiles;
    }
    if (pack_pays(tiles, packed)) return;
    for (int m = 0; m < n; ++m) set_tiles(d[m], ty[m], false);
}

inline int default_tile_rows(int nx, int ny) {
    return rows_for([=](int rows) { return grid_tiles(nx, ny, rows); }, 1);
}

// A tile next to a one-row tile at a south Chapman edge would read a ghost
// row that depends on what the edge's tile overwrites: two rows at least
// there (tile_range sees to the north edge).
inline int tile_rows_of(const rkg_grid* g) {
    const int ty = g->ty > 0 ? g->ty : default_tile_rows(g->cfg.nx, g->cfg.ny);
    bool chapman = false;
    for (int s = 0; s < 4; ++s) chapman = chapman || g->cfg.bc[s] == RKG_BC_CHAPMAN;
    return chapman && ty < 2 ? 2 : ty;
}

// apply_sponge does something (rki_kernel_sponge.F90:42-47 and a sponge edge).
inline bool sponge_on(const rkg_grid* g) {
    if (g->sponge_width <= 0 || !(g->sponge_strength > 0.0)) return false;
    for (int s = 0; s < 4; ++s)
        if (g->cfg.bc[s] == RKG_BC_SPONGE) return true;
    return false;
}

// The configuration-derived part of a descriptor for a grid of row pitch
// `pitch` and `ty` rows per tile; the buffer pointers are left null.
inline GridDesc desc_of_config(const rkg_config& c, long long pitch, int ty) {
    GridDesc d;
    memset(&d, 0, sizeof d);
    d.nx = c.nx; d.ny = c.ny; d.pitch = pitch;
    d.dx = c.dx; d.dy = c.dy;
    d.sdx = spacing(c.dx); d.sdy = spacing(c.dy);
    d.plane = pitch * (long long)c.ny;
    d.g = c.g; d.cfl = c.cfl; d.manning_n = c.manning_n; d.coriolis_f = c.coriolis_f;
    d.use_hllc = c.use_hllc;
    for (int s = 0; s < 4; ++s) d.bc[s] = c.bc[s];
    d.tidal_amplitude = c.tidal_amplitude; d.tidal_period = c.tidal_period;
    d.n_tc = c.n_tidal_constituents;
    for (int n = 0; n < RKG_MAX_TIDAL_CONSTITUENTS; ++n) {
        d.tc_amp[n] = c.tidal_amp[n]; d.tc_phase[n] = c.tidal_phase[n]; d.tc_omega[n] = c.tidal_omega[n];
    }
    d.inflow_velocity = c.inflow_velocity; d.discharge_flux = c.discharge_flux;
    d.clamped_elevation = c.clamped_elevation;
    d.dt_fixed = c.dt_fixed; d.t_end = c.t_end;
    d.cfl_interval = c.cfl_interval;
    set_launch_tiles(&d, 1, &ty);
    d.ssp_coeff = 1.0;
    return d;
}

inline GridDesc make_desc(rkg_grid* g) {
    GridDesc d = desc_of_config(g->cfg, g->pitch, tile_rows_of(g));
    d.ah = plane_ptr(g, 0); d.ahu = plane_ptr(g, 1); d.ahv = plane_ptr(g, 2);
    d.bh = plane_ptr(g, 3); d.bhu = plane_ptr(g, 4); d.bhv = plane_ptr(g, 5);
    d.bed = plane_ptr(g, 6);
    d.o2h = d.ah; d.o2hu = d.ahu; d.o2hv = d.ahv;
    d.nfield = g->nfield;
    d.rec = nullptr;
    d.sh = g->save;
    d.shu = g->save ? g->save + g->plane : nullptr;
    d.shv = g->save ? g->save + 2 * g->plane : nullptr;
    d.ctrl = g->ctrl;
    d.mpart = g->mpart;
    if (sponge_on(g)) {
        d.sponge_width = g->sponge_width;
        d.sponge_strength = g->sponge_strength;
        d.sponge_h_ref = g->sponge_h_ref;
        d.spart = g->mpart ? g->mpart + 2 * g->mpart_cap : nullptr;
    }
    if (g->forcing) {
        d.fwx = g->frc;
        d.fwy = g->frc + g->plane;
        d.frain = g->frc + 3 * g->plane;
        d.fdpx = g->frc + 4 * g->plane;
        d.fdpy = g->frc + 5 * g->plane;
    }
    d.ssp_coeff = g->scheme == RKG_TIME_RK43 ? 2.0 : 1.0;  // rki_timestepper.F90:60-100
    d.plain_rows = g->fast_mode < 0 ? 1 : 0;
    return d;
}


}  // namespace rk

#define HIP_TRY(expr)                                                          \
    do {                                                                       \
        hipError_t e_ = (expr);                                                \
        if (e_ != hipSuccess) {                                                \
            rk::set_error("%s failed: %s", #expr, hipGetErrorString(e_));      \
            return RKG_ERR_HIP;                                                \
        }                                                                      \
    } while (0)
