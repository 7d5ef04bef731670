// stage_kernels.hpp -- the stage kernels and the small reductions shared by
// the single-grid ABI (rkg_api.hip) and the ensemble ABI
// (rkg_ensemble.hip).  Kernels have internal linkage: each translation unit
// that launches them holds its own copy.
#pragma once

#include <vector>

#include "swe_kernels.hpp"

#ifndef RKG_WAVES_PER_EU
#define RKG_WAVES_PER_EU 3
#endif

namespace rk {
namespace {

constexpr int MODE_STEP = 0;
constexpr int MODE_ADVANCE = 1;
constexpr int MASS_BLOCKS = 512;

// Way `lane % SPEED_WAYS` of a slot's max CFL speed.
__device__ __forceinline__ unsigned long long speed_way(const CtrlSlot& c) {
    return c.speed[(threadIdx.x & (SPEED_WAYS - 1)) * SPEED_STRIDE];
}

template <int ROR>
__device__ __forceinline__ double row_ror(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x120 + ROR, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x120 + ROR, 0xf, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

__device__ __forceinline__ double wave_first(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readfirstlane((int)b), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// The maximum of the ways that the lanes of a row of 16 hold.
__device__ __forceinline__ double speed_max(unsigned long long way) {
    static_assert(SPEED_WAYS == 16, "one way per lane of a row");
    double v = __longlong_as_double((long long)way);
    v = dmax(v, row_ror<8>(v));
    v = dmax(v, row_ror<4>(v));
    v = dmax(v, row_ror<2>(v));
    v = dmax(v, row_ror<1>(v));
    return v;
}

__device__ __forceinline__ void speed_add(CtrlSlot& c, unsigned who, double speed) {
    atomicMax(&c.speed[(who & (SPEED_WAYS - 1)) * SPEED_STRIDE], (unsigned long long)__double_as_longlong(speed));
}

// dt of a step from the control slot of the state it starts from:
// rki_solver.F90:728-745 with rki_api.F90:377 (step) / :402 (advance).
__device__ __forceinline__ double step_dt(const GridDesc& d, const CtrlClock& cp, double max_speed, double dt_max) {
    if (d.dt_fixed > 0.0) return dmin(d.dt_fixed, dt_max);
    if (cp.step_count % d.cfl_interval == 0 || cp.dt <= 0.0) {
        double dt;
        if (max_speed > 0.0)
            dt = d.cfl / max_speed;
        else
            dt = d.cfl * dmin(d.dx, d.dy) / sqrt(d.g * DRY_TOLERANCE);
        dt = dt * d.ssp_coeff;  // rki_solver.F90:736-741
        return dmin(dt, dt_max);
    }
    return cp.dt;
}

__device__ __forceinline__ SourceTerms make_src(const GridDesc& d, double dt) {
    SourceTerms s;
    s.g = d.g;
    s.n_sq = d.manning_n * d.manning_n;
    s.has_friction = d.manning_n > 0.0;
    s.has_coriolis = fabs(d.coriolis_f) > 1.0e-20;
    s.cosf = 0.0;
    s.sinf = 0.0;
    s.coriolis_f = d.coriolis_f;
    if (s.has_coriolis) {
        s.cosf = crm::cos(d.coriolis_f * dt);
        s.sinf = crm::sin(d.coriolis_f * dt);
    }
    return s;
}

// One tile of one stage of one grid.  `where(d, leader)` gives the tile; the
// leader is the single tile per grid and launch that advances the control slot.  STAGE 1 and 2 are the fused
// SSP-RK2 stages; STAGE 3 is one stage `gs` of a generic SSP scheme.
template <int STAGE, bool HLLC, bool NF, bool REC, class Where, int FEAT = 0>
__device__ __forceinline__ void stage_tile(const GridDesc& d, TileRing& ring, int p, int mode, double tlim, Where where, const GenStage& gs = GenStage{}) {
    bool leader;
    const TileAt w = where(d, leader);
    const int strip = w.strip, seg = w.seg;
    StageCtx s;
    int x0, x1;
    tile_range(d.nx, OWN, d.nstrips, strip, x0, x1);
    tile_range(d.ny, d.ty, d.nsegs, seg, s.row0, s.row1);   // of several segments, those of the first
    const bool west = x0 < HALO, east = x0 + OWN + HALO > d.nx;
    const bool south = s.row0 < HALO, north = s.row1 + HALO > d.ny;
    const bool edge = west || east || south || north;
    // the stage's input and the first rows of the march, before the clock
    if (STAGE == 1) { s.ih = d.ah; s.ihu = d.ahu; s.ihv = d.ahv; }
    else if (STAGE == 2) { s.ih = d.bh; s.ihu = d.bhu; s.ihv = d.bhv; }
    else { s.ih = gs.ih; s.ihu = gs.ihu; s.ihv = gs.ihv; }
    const TileLane lane = edge ? tile_lane<true>(d, w, x0, x1, threadIdx.x) : tile_lane<false>(d, w, x0, x1, threadIdx.x);
    const FirstRows first = edge ? first_rows<true>(d, s, lane, s.row0) : first_rows<false>(d, s, lane, s.row0);
    s.alpha = 0.0; s.a_prev = 1.0;
    s.blend = false; s.first = false; s.last = false;
    s.radiate = false; s.prev_h = nullptr; s.bc_dt = 0.0;
    s.eta_tidal = 0.0;
    double t_tide;   // bc%time of the stage; the tide is evaluated by edge tiles only
    if (STAGE == 1 || (STAGE == 3 && gs.first)) {
        const CtrlClock cp = d.ctrl[p];
        const unsigned long long way = speed_way(d.ctrl[p]);
        const bool active = (mode == MODE_STEP) || (cp.t < tlim - 1.0e-10);
        const double dt_max = tlim - cp.t;
        const double dt = active ? wave_first(step_dt(d, cp, speed_max(way), dt_max)) : cp.dt;
        if (leader && threadIdx.x < SPEED_WAYS) d.ctrl[1 - p].speed[threadIdx.x * SPEED_STRIDE] = active ? 0ull : way;
        if (leader && threadIdx.x == 0) {
            CtrlClock* q = &d.ctrl[1 - p];
            q->t = active ? cp.t + dt : cp.t;
            q->dt = dt;
            q->step_count = active ? cp.step_count + 1 : cp.step_count;
            q->mass_out = cp.mass_out;
            q->mass_src = cp.mass_src;
            q->active = active ? 1 : 0;
            // the last boundary call: stage 2 at t + dt, or the last generic
            // stage at t + c_last dt (rki_solver.F90:790-795, :895-897)
            if (!active) q->t_bc = cp.t_bc;
            else if (STAGE == 1) q->t_bc = cp.t + dt;
            else q->t_bc = cp.t + gs.c_last * dt;
            if (REC && d.hist != nullptr) {   // the step's clock for a reverse sweep (rki_solver.F90:731)
                d.hist[0] = cp.t;
                d.hist[1] = dt;
                d.hist[2] = (d.dt_fixed <= 0.0 && (cp.step_count % d.cfl_interval == 0 || cp.dt <= 0.0)) ? 1.0 : 0.0;
            }
        }
        if (!active) return;
        s.bc_dt = dt;   // bc%dt = state%dt, rki_solver.F90:748
        if (STAGE == 1) {
            s.oh = d.bh; s.ohu = d.bhu; s.ohv = d.bhv;
            s.dt = dt;
        } else {
            s.oh = gs.oh; s.ohu = gs.ohu; s.ohv = gs.ohv;
            s.dt = gs.beta * dt;
        }
        t_tide = cp.t;  // stage abscissa c_1 = 0
    } else if (STAGE == 3) {
        const CtrlClock cp = d.ctrl[p];
        const CtrlClock cq = d.ctrl[1 - p];
        if (!cq.active) return;
        s.oh = gs.oh; s.ohu = gs.ohu; s.ohv = gs.ohv;
        s.dt = gs.beta * cq.dt;
        t_tide = cp.t + gs.c * cq.dt;  // bc%time = t_base + c_i dt
        s.bc_dt = cq.dt;
        s.radiate = true;       // against the previous stage's input
        s.prev_h = gs.ph;
    } else {
        const CtrlClock cq = d.ctrl[1 - p];
        if (!cq.active) return;
        s.oh = d.o2h; s.ohu = d.o2hu; s.ohv = d.o2hv;
        s.dt = cq.dt;
        t_tide = cq.t;  // bc%time = t + dt
        s.bc_dt = cq.dt;
        s.radiate = true;       // against U^n, the input of stage 1
        s.prev_h = d.ah;
    }
    if (STAGE == 3) {
        s.alpha = gs.alpha;
        s.a_prev = 1.0 - gs.alpha;
        s.blend = gs.alpha != 0.0;
        s.first = gs.first != 0;
        s.last = gs.last != 0;
    }
    s.src = make_src(d, s.dt);
    double smax, fsum, ssum;
    if (!edge) {
        const TileLane inner = tile_lane<false>(d, w, x0, x1, threadIdx.x);   // again, not kept through the clock's code
        smax = process_tile<STAGE, HLLC, false, NF, REC, FEAT>(d, s, ring, inner, first, s.row0, s.row1, fsum, ssum);
    } else {
        // the tide (a correctly rounded sine, a long dependent chain) only
        // where the tile reads ghost cells of a tidal edge
        if ((west && d.bc[0] == BC_TIDAL) || (east && d.bc[1] == BC_TIDAL) || (south && d.bc[2] == BC_TIDAL) ||
            (north && d.bc[3] == BC_TIDAL))
            s.eta_tidal = tidal_eta(d, t_tide);
        smax = process_tile<STAGE, HLLC, true, NF, REC, FEAT>(d, s, ring, lane, first, s.row0, s.row1, fsum, ssum);
    }
    if (STAGE == 2 || STAGE == 3) {
        smax = wave_max(smax);
        if (threadIdx.x == 0 && smax > 0.0) speed_add(d.ctrl[1 - p], (unsigned)(strip + seg * d.nstrips), smax);
    }
    // the sums of a tile go to its first segment's slot, zeros to the other segments'
    const int slots = d.nstrips * d.nsegs;
    const long long slot = (long long)(STAGE - 1) * slots + (long long)(seg + (int)threadIdx.x) * d.nstrips + strip;
    if (STAGE != 3 && d.mpart != nullptr) {  // accumulate_boundary_mass_out's sum, per tile
        fsum = wave_sum(fsum);
        if ((int)threadIdx.x < w.count) d.mpart[slot] = threadIdx.x == 0 ? fsum : 0.0;
    }
    if ((FEAT & FEAT_SPONGE) && STAGE != 3 && d.spart != nullptr) {  // accumulate_sponge_mass_src
        ssum = wave_sum(ssum);
        if ((int)threadIdx.x < w.count) d.spart[slot] = threadIdx.x == 0 ? ssum : 0.0;
    }
}

// Single grid: one workgroup (one wavefront) per tile.
struct SingleGridTile {
    __device__ TileAt operator()(const GridDesc& g, bool& leader) const {
        leader = blockIdx.x == 0;
        return tile_at(g, xcd_tile(blockIdx.x, g.ntiles));
    }
};

// A tile of one member of a batch, as the tables list them.
struct BatchTile {
    int member, strip, seg, count;   // count negative: the leader
    __device__ TileAt operator()(const GridDesc&, bool& leader) const {
        leader = count < 0;
        return TileAt{strip, seg, leader ? -count : count};
    }
};

// Member m's tiles, in the order and with the leader of its own launches.
inline void batch_tiles(const GridDesc& d, int m, std::vector<BatchTile>& t) {
    for (int k = 0; k < d.ntiles; ++k) {
        const TileAt w = tile_at(d, k);
        t.push_back(BatchTile{m, w.strip, w.seg, k == 0 ? -w.count : w.count});
    }
}

// FEAT: FEAT_FORCING / FEAT_SPONGE / FEAT_CHAPMAN source terms.
template <int STAGE, bool HLLC, bool NF, bool REC, int FEAT = 0>
__global__ __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(RKG_WAVES_PER_EU, 8))) void k_stage(GridDesc d, int p, int mode, double tlim) {
    __shared__ TileRing ring;
    stage_tile<STAGE, HLLC, NF, REC, SingleGridTile, FEAT>(d, ring, p, mode, tlim, SingleGridTile{});
}

// One stage of a generic SSP scheme, single grid.
template <bool HLLC, bool NF, int FEAT = 0>
__global__ __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(RKG_WAVES_PER_EU, 8))) void k_stage_gen(GridDesc d, GenStage gs, int p, int mode, double tlim) {
    __shared__ TileRing ring;
    stage_tile<3, HLLC, NF, false, SingleGridTile, FEAT>(d, ring, p, mode, tlim, SingleGridTile{}, gs);
}

// Resets control slot p to time t / step count n with an empty speed max;
// the mass budget is set to mass_out.  One workgroup of 64 threads.
__global__ void k_ctrl_reset(CtrlSlot* ctrl, int p, double t, double dt, long long n, double mass_out,
                             double mass_src) {
    if (threadIdx.x < SPEED_WAYS) ctrl[p].speed[threadIdx.x * SPEED_STRIDE] = 0ull;
    if (threadIdx.x == 0) {
        ctrl[p].t = t;
        ctrl[p].dt = dt;
        ctrl[p].step_count = n;
        ctrl[p].mass_out = mass_out;
        ctrl[p].mass_src = mass_src;
        ctrl[p].active = 1;
        ctrl[p].t_bc = t;
    }
}

// k_ctrl_reset to the slot's own clock and budget.
__global__ void k_speed_reset(CtrlSlot* ctrl, int p) {
    if (threadIdx.x < SPEED_WAYS) ctrl[p].speed[threadIdx.x * SPEED_STRIDE] = 0ull;
    if (threadIdx.x == 0) {
        ctrl[p].active = 1;
        ctrl[p].t_bc = ctrl[p].t;
    }
}

// Boundary mass budget of one SSP-RK2 step (rki_solver.F90:507-537, called
// after each stage's flux at :769 and :796): mass_out -= 0.5 dt sum(flux_h)
// area per stage.  The per-tile sums of both stages are added in a fixed
// order (strided per thread, then a tree).  mass_src, per stage and in
// the reference's order: with the surface forcing on, `rain` holds the
// interior sum of the precipitation rate and mass_src += 0.5 dt rain area
// (accumulate_mass_src, rki_solver.F90:539-606, at :783 and :810); with the
// sponge on, `spart` holds the per-tile sums of its change of h and
// mass_src += 0.5 sum area (accumulate_sponge_mass_src, :608-657, at :787
// and :814).  Slot 1-p is the step's result.
__device__ __forceinline__ void step_budget(const BudgetArgs& b) {
    __shared__ double red[4][256];
    CtrlSlot* ctrl = b.ctrl;
    const int p = b.p, ntiles = b.ntiles;
    const double *mpart = b.mpart, *rain = b.rain, *spart = b.spart;
    const double area = b.area;
    if (!ctrl[1 - p].active) return;
    double a[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int i = threadIdx.x; i < ntiles; i += 256) {
        a[0] = a[0] + mpart[i];
        a[1] = a[1] + mpart[ntiles + i];
        if (spart != nullptr) {
            a[2] = a[2] + spart[i];
            a[3] = a[3] + spart[ntiles + i];
        }
    }
    for (int q = 0; q < 4; ++q) red[q][threadIdx.x] = a[q];
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s)
            for (int q = 0; q < 4; ++q) red[q][threadIdx.x] = red[q][threadIdx.x] + red[q][threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        CtrlSlot* q = &ctrl[1 - p];
        const double dt = q->dt;
        double m = q->mass_out;
        m = m - 0.5 * dt * red[0][0] * area;
        m = m - 0.5 * dt * red[1][0] * area;
        q->mass_out = m;
        double src = q->mass_src;
        for (int st = 0; st < 2; ++st) {
            if (rain != nullptr) src = src + 0.5 * dt * (*rain) * area;
            if (spart != nullptr) src = src + 0.5 * red[2 + st][0] * area;
        }
        q->mass_src = src;
    }
}

__global__ __launch_bounds__(256) void k_budget(BudgetArgs b) { step_budget(b); }

// Max CFL speed over all cells, whose states load(offset, h, hu, hv) gives;
// the result is valid in thread 0.  Workgroups of 256 threads, cell after cell
// with the grid as stride, row and column kept without divisions.
template <class LOAD>
__device__ __forceinline__ double plane_speed(const GridDesc& d, LOAD load) {
    __shared__ double red[4];
    const long long stride = (long long)gridDim.x * 256, k = blockIdx.x * 256ll + threadIdx.x;
    const int dj = (int)(stride / d.nx), di = (int)(stride % d.nx);
    int j = (int)(k / d.nx), i = (int)(k % d.nx);
    double m = 0.0;
    while (j < d.ny) {
        double h, hu, hv;
        load((long long)j * d.pitch + i, h, hu, hv);
        m = dmax(m, cfl_speed(d.g, d.dx, d.dy, h, hu, hv));
        i += di; j += dj;
        if (i >= d.nx) { i -= d.nx; ++j; }
    }
    m = wave_max(m);
    if ((threadIdx.x & (WAVE - 1)) == 0) red[threadIdx.x / WAVE] = m;
    __syncthreads();
    return dmax(dmax(red[0], red[1]), dmax(red[2], red[3]));
}

// End of a one-stage (Euler) step: the stage wrote B, so B is copied to A
// and the CFL max of the new state goes to slot 1-p.  (The stage kernel
// cannot take that max itself: its leader clears the slot's max while the
// other tiles of the same launch run.)
__global__ __launch_bounds__(256) void k_euler_finish(GridDesc d, int p) {
    if (!d.ctrl[1 - p].active) return;
    const double m = plane_speed(d, [&](long long o, double& h, double& hu, double& hv) {
        h = d.bh[o]; hu = d.bhu[o]; hv = d.bhv[o];
        d.ah[o] = h; d.ahu[o] = hu; d.ahv[o] = hv;
    });
    if (threadIdx.x == 0 && m > 0.0) speed_add(d.ctrl[1 - p], blockIdx.x, m);
}

// Max CFL speed of the state A into slot p (compute_timestep's reduction,
// rki_kernel_timestep.F90:53-70).  One atomic per workgroup, spread over the
// slot's ways: the 16384 atomics of one per wavefront on one address took
// 190 us at 1024x1024 and more; the sweep now takes 12.
__global__ __launch_bounds__(256) void k_init_speed(GridDesc d, int p) {
    const double m = plane_speed(d, [&](long long o, double& h, double& hu, double& hv) {
        h = d.ah[o]; hu = d.ahu[o]; hv = d.ahv[o];
    });
    if (threadIdx.x == 0 && m > 0.0) speed_add(d.ctrl[p], blockIdx.x, m);
}

// Workgroups of a sweep over all cells: 1024 (four per CU) cover the chip.
inline int sweep_blocks(long long cells) { return (int)((cells + 255) / 256 < 1024 ? (cells + 255) / 256 : 1024); }

// Mass partials: block b sums rows b, b + gridDim.x, ... in a fixed order
// (compute_total_mass, rki_init.F90:287-317).
__global__ __launch_bounds__(256) void k_mass_partial(GridDesc d, double* partial) {
    __shared__ double red[256];
    const double area = d.dx * d.dy;
    double acc = 0.0;
    for (int j = blockIdx.x; j < d.ny; j += gridDim.x) {
        for (int i = threadIdx.x; i < d.nx; i += 256) {
            const double h = d.ah[(long long)j * d.pitch + i];
            if (h > 0.0 && h < 1.0e6) acc = acc + h * area;
        }
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] = red[threadIdx.x] + red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// The central pressure gradient of the surface forcing
// (rki_kernel_fused.F90:277-278), dp/dx = (p(i+1) - p(i-1)) / (2 dx), with
// pressure 0 outside the grid (the ghost cells, which no setter writes);
// computed once per pressure field, in the same operations as per stage.
__global__ __launch_bounds__(256) void k_pressure_gradient(const double* p, double* dpx, double* dpy, int nx,
                                                           int ny, long long pitch, double dx, double dy) {
    const long long n = (long long)nx * ny;
    for (long long q = blockIdx.x * 256ll + threadIdx.x; q < n; q += (long long)gridDim.x * 256) {
        const int c = (int)(q % nx), j = (int)(q / nx);
        const long long k = (long long)j * pitch + c;
        const double pe = c + 1 < nx ? p[k + 1] : 0.0;
        const double pw = c > 0 ? p[k - 1] : 0.0;
        const double pn = j + 1 < ny ? p[k + pitch] : 0.0;
        const double ps = j > 0 ? p[k - pitch] : 0.0;
        dpx[k] = (pe - pw) / (2.0 * dx);
        dpy[k] = (pn - ps) / (2.0 * dy);
    }
}

// Per-block sums of the interior of one plane (rows strided over blocks),
// added up by k_mass_final: a fixed order, so the result is deterministic.
__global__ __launch_bounds__(256) void k_plane_sum_partial(const double* f, long long pitch, int nx, int ny,
                                                           double* partial) {
    __shared__ double red[256];
    double acc = 0.0;
    for (int j = blockIdx.x; j < ny; j += gridDim.x)
        for (int i = threadIdx.x; i < nx; i += 256) acc = acc + f[(long long)j * pitch + i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] = red[threadIdx.x] + red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void k_mass_final(const double* partial, int n, double* out) {
    __shared__ double red[256];
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) acc = acc + partial[i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] = red[threadIdx.x] + red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = red[0];
}

}  // namespace
}  // namespace rk
