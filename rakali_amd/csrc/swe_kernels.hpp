// swe_kernels.hpp -- device-side data layout, ghost-cell synthesis and the
// strip-marching tile routine shared by the single-grid stage kernels.
//
// Layout in HBM: structure of arrays, one FP64 plane per field, row-major
// with x fastest (the reference's column-major (i, j) order), interior cells
// only, row pitch `pitch` elements (a multiple of 16, i.e. 128-byte rows).
// State buffers: A = U^n (h, hu, hv; overwritten in place by U^{n+1}),
// B = U* (stage-1 output), and the bed b.  Ghost cells are never stored:
// the tile loader synthesizes them from the boundary tags exactly as
// apply_boundary_conditions (rki_boundary.F90:40-470) would have filled
// them for the rows and columns the cross-shaped stencil reads.
#pragma once

#include "swe_core.hpp"

namespace rk {

constexpr int WAVE = 64;        // wavefront width on CDNA
constexpr int MAX_TC = 10;      // MAX_TIDAL_CONSTITUENTS
// Time-control slot.  Two slots ping-pong: a step reads slot p (state at
// the start of the step) and its stage-1 kernel writes slot 1-p.
struct CtrlClock {
    double t;                     // time at the start of the step
    double dt;                    // dt of the step that produced this slot
    long long step_count;         // state%step_count
    double mass_out;              // boundary mass budget (rki_solver.F90:507-537)
    int active;                   // 1 if the step that wrote this slot ran
    int pad;
    double mass_src;              // surface mass source (accumulate_mass_src, rki_solver.F90:539-606)
    double t_bc;                  // bc%time of the step's last boundary call
};

// The clock and the max CFL speed of its state, as the bits of positive
// doubles.  Atomics on one address complete one after the other, 12 ns apart
// (16384 of them take 190 us): the tiles of a launch spread theirs over
// SPEED_WAYS cache lines, and a reader takes the maximum of the ways.
constexpr int SPEED_WAYS = 16;
constexpr int SPEED_STRIDE = 16;  // 128 bytes

struct alignas(128) CtrlSlot : CtrlClock {
    alignas(128) unsigned long long speed[SPEED_WAYS * SPEED_STRIDE];
};

// Arguments of a step's mass budget (k_budget); mpart null: none.
struct BudgetArgs {
    CtrlSlot* ctrl;
    int p;
    const double* mpart;
    int ntiles;
    double area;
    const double* rain;
    const double* spart;
};

// Optional source terms of the stage kernels (template bit mask).
constexpr int FEAT_FORCING = 1;   // surface forcing, rki_kernel_fused.F90:268-289
constexpr int FEAT_SPONGE = 2;    // sponge relaxation, rki_kernel_sponge.F90:16-88
constexpr int FEAT_CHAPMAN = 4;   // Chapman radiation edges, rki_boundary.F90:471-552

struct GridDesc {
    int nx, ny;
    long long pitch;              // elements per row
    double dx, dy;
    Spacing sdx, sdy;             // dx and dy as divisors
    double* ah; double* ahu; double* ahv;   // A: U^n / U^{n+1}
    double* bh; double* bhu; double* bhv;   // B: U*
    double* sh; double* shu; double* shv;   // optional copy of U^n (RK save), or null
    double* o2h; double* o2hu; double* o2hv; // stage-2 output (normally A itself)
    const double* bed;
    const double* nfield;         // per-cell Manning n, or null (scalar manning_n)
    double* rec;                  // 3 planes receiving each cell's flux divergence, or null
    double* mpart;                // per-tile sums of flux_h, [stage 1 tiles | stage 2 tiles], or null
    double* hist;                 // recording stage 1: (t, dt, dt recomputed) of the step, or null
    const double* fwx; const double* fwy;   // surface forcing planes (FEAT_FORCING kernels): wind
    const double* fdpx; const double* fdpy; // stress, the central pressure gradient (from the
    const double* frain;                    // pressure field, see k_pressure_gradient), precipitation
    double* spart;                // per-tile sums of the sponge's h change, [stage 1 | stage 2], or null
    int sponge_width;             // sponge relaxation band (FEAT_SPONGE kernels), bc_params_t
    double sponge_strength, sponge_h_ref;
    long long plane;              // elements per plane (pitch * ny)
    double ssp_coeff;             // stable-dt multiplier of the time scheme (rki_timestepper.F90)
    double g, cfl, manning_n, coriolis_f;
    int use_hllc;
    int bc[4];                    // west, east, south, north
    double tidal_amplitude, tidal_period;
    int n_tc;
    double tc_amp[MAX_TC], tc_phase[MAX_TC], tc_omega[MAX_TC];
    double inflow_velocity, discharge_flux, clamped_elevation;
    double dt_fixed, t_end;
    int cfl_interval;
    int ty;                       // rows per tile segment (<= 64)
    int plain_rows;               // every row with plain divisions (rkg_set_fast_path(-1))
    int nstrips, nsegs;
    int ntiles;                   // wavefronts of a launch, see tile_at
    unsigned strips_inv;          // 2^32 / nstrips, rounded up (0 for one strip)
    int pack, pack_seg, pack_n;   // segments of the last strip that share a wavefront (1: none); the
                                  // first and the number of the segments that do
    CtrlSlot* ctrl;               // [2]
};

// Tidal surface, rki_boundary.F90:92-101.
__host__ __device__ __forceinline__ double tidal_eta(const GridDesc& d, double time) {
    double e = 0.0;
    if (d.n_tc > 0) {
        for (int n = 0; n < d.n_tc; ++n) e = e + d.tc_amp[n] * crm::cos(d.tc_omega[n] * time - d.tc_phase[n]);
    } else if (d.tidal_period > 0.0) {
        e = d.tidal_amplitude * crm::sin(TWO_PI * time / d.tidal_period);
    }
    return e;
}

// A pointer into device memory, which the compiler otherwise knows only of
// kernel arguments taken by value.  Through a pointer that was itself loaded
// (a batch's descriptors) it would use flat accesses, which the LDS counter
// counts too: every LDS read of a row then waited for the next row's loads
// (ensembles of 64 x 256^2, 32 x 512..1024^2: 306 -> 302, 1239 -> 1220 us a step).
template <class T>
__device__ __forceinline__ T __attribute__((address_space(1)))* in_hbm(T* p) {
    return (T __attribute__((address_space(1)))*)p;
}

__device__ __forceinline__ Cell load_direct(const double* __restrict__ h, const double* __restrict__ hu,
                                            const double* __restrict__ hv, const double* __restrict__ b,
                                            long long pitch, int c, int j) {
    const long long k = (long long)j * pitch + c;
    Cell r;
    r.h = in_hbm(h)[k]; r.hu = in_hbm(hu)[k]; r.hv = in_hbm(hv)[k]; r.b = in_hbm(b)[k];
    return r;
}

// Ghost value for an edge, from the interior cells along its normal.
// `nrm_sign` is -1 on W/S and +1 on E/N; `normal_is_u` on W/E.
// kk = ghost layer (0 = adjacent), mir = mirror cell for wall edges,
// in0 = first interior cell.  rki_boundary.F90:220-466.
__host__ __device__ __forceinline__ Cell ghost_from(const GridDesc& d, int tag, double eta_tidal,
                                           const Cell& mir, const Cell& in0, double nrm_sign,
                                           bool normal_is_u) {
    Cell g;
    switch (tag) {
    case BC_WALL:
    case BC_SPONGE: {   // bc_wall_edge :281-289 (bed mirrored first)
        g.b = mir.b;
        g.h = fmax0(mir.h + mir.b - g.b);
        if (normal_is_u) { g.hu = -mir.hu; g.hv = mir.hv; }
        else { g.hv = -mir.hv; g.hu = mir.hu; }
        return g;
    }
    case BC_OPEN:
    case BC_TIDAL: {    // bc_flather_edge :331-343; bed ghost = first interior
        const bool prescribe = (tag == BC_TIDAL);
        const double eta_ext = prescribe ? eta_tidal : 0.0;
        g.b = in0.b;
        const double h_int = in0.h;
        const double eta_int = h_int + in0.b;
        const double hmax = dmax(h_int, 1.0e-6);
        const double speed = sqrt(d.g * hmax);
        const double h_ghost = prescribe ? fmax0(eta_ext - g.b) : h_int;
        g.h = h_ghost;
        const double nrm = normal_is_u ? in0.hu : in0.hv;
        const double rad = h_ghost * (nrm / hmax + nrm_sign * speed * (eta_int - eta_ext) / hmax);
        if (normal_is_u) { g.hu = rad; g.hv = in0.hv; }
        else { g.hv = rad; g.hu = in0.hu; }
        return g;
    }
    case BC_INFLOW:
    case BC_DISCHARGE: {  // bc_inflow_edge :377-387, bc_disch_edge :418-428
        const double in_sgn = -nrm_sign;
        g.b = in0.b;
        g.h = in0.h;
        const double nrm = (tag == BC_INFLOW) ? in_sgn * in0.h * d.inflow_velocity
                                              : in_sgn * d.discharge_flux;
        if (normal_is_u) { g.hu = nrm; g.hv = in0.hv; }
        else { g.hv = nrm; g.hu = in0.hu; }
        return g;
    }
    case BC_CLAMPED:
    default: {          // bc_clamped_edge :458-464
        g.b = in0.b;
        g.h = fmax0(d.clamped_elevation - g.b);
        g.hu = in0.hu;
        g.hv = in0.hv;
        return g;
    }
    }
}

// Workgroup id -> tile id so that each XCD (workgroups are dispatched to
// the 8 XCDs round-robin) owns one contiguous band of tiles and the halo
// rows and columns it shares stay in that XCD's L2.
__device__ __forceinline__ int xcd_tile(int b, int n) {
    const int x = b & 7, k = b >> 3;
    const int per = n >> 3, rem = n & 7;
    return x * per + (x < rem ? x : rem) + k;
}

__device__ __forceinline__ double shfl_down1(double v) { return __shfl_down(v, 1, WAVE); }
__device__ __forceinline__ double shfl_up1(double v) { return __shfl_up(v, 1, WAVE); }

__device__ __forceinline__ FState shfl_down1(const FState& x) {
    return FState{shfl_down1(x.h), shfl_down1(x.hu), shfl_down1(x.hv)};
}

__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = dmax(v, __shfl_xor(v, off, WAVE));
    return v;
}

// Butterfly sum: every lane ends with the same bits (each pairwise add sees
// the same two operands), in an order fixed by the lane numbering.
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = v + __shfl_xor(v, off, WAVE);
    return v;
}

// Orders the LDS writes of one wavefront's lanes before the reads of its other
// lanes (and those reads before the next writes).  A wavefront's LDS accesses
// are performed in order, so it is no instruction; it keeps the compiler from
// moving them, which per lane it may (the addresses of two lanes differ).
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// Three rows of the march, (h + b, hu, hv, b, h) of the wavefront's 64
// columns, and what the row below hands up: its high y state (h, hu, hv), the
// part of its upper face that the row above takes (fh, fhu, fhv, a) and the
// differences across that face (h + b, hu, hv).  12.5 KB: 12 wavefronts, three
// a SIMD, on a CU's 160 KB.
struct TileRing {
    double v[3][5][WAVE];
    double up[10][WAVE];
};

struct StageCtx {
    const double* ih; const double* ihu; const double* ihv;   // stage input
    double* oh; double* ohu; double* ohv;                     // stage output
    double dt;
    double eta_tidal;
    SourceTerms src;
    // Chapman edges (FEAT_CHAPMAN): whether this boundary call radiates
    // (its state differs from the previous call's), the previous call's
    // state prev_h (its eta_old = prev_h + b at the first interior cell),
    // the step's dt (bc%dt) and the own rows of the tile's first segment
    bool radiate;
    const double* prev_h;
    double bc_dt;
    int row0, row1;
    // generic SSP stage only (STAGE 3)
    double alpha, a_prev;         // blend weights on U^n and on the Euler iterate
    bool blend, first, last;
};

// One stage of a generic explicit SSP scheme (rki_solver.F90:861-925):
// E = U^(i-1) + beta_i dt L(U^(i-1)), then U^(i) = alpha_i U^n +
// (1 - alpha_i) E when alpha_i != 0.  U^n stays in A until the last stage,
// which writes A.
struct GenStage {
    const double* ih; const double* ihu; const double* ihv;
    double* oh; double* ohu; double* ohv;
    const double* ph;             // h of the previous stage's input (Chapman eta_old), or null
    double alpha, beta, c;        // rki_timestepper.F90:53-58
    double c_last;                // c of the scheme's last stage (bc%time of its last call)
    int first, last;
};

// Ghost cell (c, j) of a Chapman edge (bc_chapman_edge, rki_boundary.F90:
// 471-552).  The reference calls the boundary before the dt computation
// (rki_solver.F90:718-720) and before each stage; each call sets eta_old
// to the interior eta of the state it sees (on the k = 1 layer, before the
// k = 2 layer of the same t reads it: t outer, k inner, the serial order of
// the reference's CPU build).  So
// * the first stage of a step sees eta_old = its own interior eta: the
//   ghost surface is the interior eta (the radiation term vanishes);
// * a later stage radiates on the adjacent layer against the previous
//   call's state, U^n for SSP-RK2 stage 2, the previous stage's input for
//   the generic schemes, with the step's dt; the outer layer again sees
//   eta_old = its interior eta.
// The bed ghost is the first interior bed (fill_bathymetry_ghosts_array).
// x-edge ghosts of rows outside the tile's own (own_row) are never used (the y
// pipeline loads them for lanes past the grid); they skip the radiation,
// whose eta_old the owning tile may be overwriting in place.
__device__ __forceinline__ Cell chapman_ghost(const GridDesc& d, const StageCtx& s, int side, int c, int j, bool own_row) {
    const bool xedge = side < 2, lo = (side & 1) == 0;
    const int kk = xedge ? (lo ? -c - 1 : c - d.nx) : (lo ? -j - 1 : j - d.ny);
    Cell g;
    g.h = 0.0; g.hu = 0.0; g.hv = 0.0; g.b = 0.0;
    if (kk > 1) return g;
    int ci = c, ji = j, c2 = c, j2 = j;
    if (xedge) { ci = lo ? 0 : d.nx - 1; c2 = lo ? 1 : d.nx - 2; }
    else { ji = lo ? 0 : d.ny - 1; j2 = lo ? 1 : d.ny - 2; }
    const Cell in0 = load_direct(s.ih, s.ihu, s.ihv, d.bed, d.pitch, ci, ji);
    const double h_int = in0.h;
    const double eta_int = h_int + in0.b;
    const double hmax = dmax(h_int, 1.0e-6);
    const double speed = sqrt(d.g * hmax);
    double eta_g = eta_int;
    if (kk == 0 && s.radiate && s.bc_dt > 0.0 && (own_row || !xedge)) {
        const long long k0 = (long long)ji * d.pitch + ci;
        const long long k2 = (long long)j2 * d.pitch + c2;
        const double dd = xedge ? d.dx : d.dy;
        const double eta_old = s.prev_h[k0] + d.bed[k0];
        const double deta_dt = (eta_int - eta_old) / s.bc_dt;
        const double deta_dx = (s.ih[k2] + d.bed[k2] - eta_int) / dd;
        double cp = fabs(deta_dx) > 1.0e-10 ? -deta_dt / deta_dx : 0.0;
        cp = dmax(0.0, fmin(cp, speed));
        eta_g = eta_old - cp * s.bc_dt / dd * (eta_old - eta_int);
    }
    g.b = in0.b;
    g.h = fmax0(eta_g - g.b);
    const double sgn = lo ? -1.0 : 1.0;
    const double nrm = xedge ? in0.hu : in0.hv;
    const double rad = g.h * (nrm / hmax + sgn * speed * (eta_int - eta_g) / hmax);
    if (xedge) { g.hu = rad; g.hv = in0.hv; }
    else { g.hv = rad; g.hu = in0.hu; }
    return g;
}

// Where a tile's lane takes its cells from.  A ghost cell depends on one cell
// of the grid, the mirror cell at a wall and the first interior cell at every
// other edge (bc_wall_edge, bc_flather_edge, ..., rki_boundary.F90:281-464),
// so each lane loads one cell a row whether it is a ghost or not, and the
// edge's rule is arithmetic on that cell.
struct LaneSource {
    int c;      // column to load
    int side;   // 0 W, 1 E: a ghost column; -1: a column of the grid; -2: beyond the ghosts
};

__host__ __device__ __forceinline__ bool mirrors(int tag) { return tag == BC_WALL || tag == BC_SPONGE; }

template <bool EDGE>
__host__ __device__ __forceinline__ LaneSource lane_source(const GridDesc& d, int c) {
    if (!EDGE || ((unsigned)c < (unsigned)d.nx)) return LaneSource{c, -1};
    const bool west = c < 0;
    const int kk = west ? -c - 1 : c - d.nx;
    if (kk > 1) return LaneSource{d.nx - 1, -2};
    const int in = mirrors(d.bc[west ? 0 : 1]) ? kk : 0;
    return LaneSource{west ? in : d.nx - 1 - in, west ? 0 : 1};
}

// A lane of a tile: its column c, the rows `row` by which its segment lies
// above the tile's first one (tiles that hold several, see tile_at), and `at`,
// the offset of its source column in the tile's row 0 of a plane (of its own
// column where it owns one).  own: its cells are the tile's; use_x: its
// right face is used.
struct TileLane {
    int c, row, side;             // side as in LaneSource
    long long at;
    bool own, use_x;
};

// The cells that row j of the march is made from: those of row j, or of the
// source row of a ghost row.
template <bool EDGE>
__device__ __forceinline__ Cell row_source(const GridDesc& d, const StageCtx& s, const TileLane& l, int j) {
    int js = j;
    if (EDGE) {
        if (j < 0) js = mirrors(d.bc[2]) ? -j - 1 : 0;
        else if (j >= d.ny) js = mirrors(d.bc[3]) ? 2 * d.ny - 1 - j : d.ny - 1;
    }
    const long long k = (long long)js * d.pitch + l.at;
    return Cell{in_hbm(s.ih)[k], in_hbm(s.ihu)[k], in_hbm(s.ihv)[k], in_hbm(d.bed)[k]};
}

// Row j of the march at the lane's column from its source cell.
template <bool EDGE, int FEAT>
__device__ __forceinline__ Cell row_cell(const GridDesc& d, const StageCtx& s, const TileLane& l, int j,
                                         const Cell& src) {
    if (!EDGE) return src;
    const int rs = j < 0 ? 2 : (j >= d.ny ? 3 : -1);
    if (rs < 0 && l.side == -1) return src;
    // corner cells and columns beyond the ghosts are not read by the stencil
    const int side = rs >= 0 ? (l.side == -1 ? rs : -2) : l.side;
    if (side < 0) return Cell{0.0, 0.0, 0.0, 0.0};
    if constexpr ((FEAT & FEAT_CHAPMAN) != 0)
        if (d.bc[side] == BC_CHAPMAN) return chapman_ghost(d, s, side, l.c, j + l.row, j >= s.row0 && j < s.row1);
    return ghost_from(d, d.bc[side], s.eta_tidal, src, src, (side & 1) ? 1.0 : -1.0, side < 2);
}

template <bool B>
struct ExactTag {
    static constexpr bool value = B;
};

// Columns of a strip that are owned and written: the wavefront's 64 lanes
// less two halo lanes on each side.
constexpr int HALO = 2;
constexpr int OWN = WAVE - 2 * HALO;

// Own range [lo, hi) of block s when [0, n) is cut into nb blocks of w, the
// last block holding at least two cells: the halo of the block before it
// then ends inside the grid, so a ghost cell (which may depend on what the
// edge's own tile overwrites, see chapman_ghost) is read by the edge's own
// tile only.  Blocks of one cell, which grids with such edges do not use, stay
// that (a last block of two would last as long as two rows: 130x97, 25 us a
// step, 21 so).
__host__ __device__ __forceinline__ void tile_range(int n, int w, int nb, int s, int& lo, int& hi) {
    lo = s * w;
    hi = lo + w < n ? lo + w : n;
    if (w >= 2 && nb >= 2 && n - (nb - 1) * w == 1) {
        if (s == nb - 1) lo = n - 2;
        if (s == nb - 2) hi = n - 2;
    }
}

// The source cells of rows j0-2 .. j0+1, loaded before the step's clock is
// read (they do not depend on it): two memory round trips in one.
struct FirstRows {
    Cell r[4];
};

// The tile `t` of a launch: `count` segments from `seg` of a strip.
struct TileAt {
    int strip, seg, count;
};

// A last strip of w <= 28 columns would leave most lanes of its wavefronts
// idle: 64 columns took the time of 120.  There `pack` = 64 / (w + 4) segments
// that lie above each other share a wavefront, each with its own halo lanes;
// they march together, so they must be of one height and touch neither the
// south nor the north ghost rows (segments pack_seg .. pack_seg + pack_n).  The
// order stays by rows, a shared wavefront after the strips beside it: at the
// end of the launch they were one XCD's alone.
__host__ __device__ __forceinline__ TileAt tile_at(const GridDesc& d, unsigned t) {
    const unsigned strips = d.nstrips, full = strips - 1, below = d.pack_seg * strips;
    unsigned seg0 = 0;
    if (__builtin_expect(d.pack > 1, 0) && t >= below) {
        t -= below;
        const unsigned per = d.pack * full + 1, group = t / per, r = t - group * per;
        const int seg = d.pack_seg + (int)group * d.pack;
        const int left = d.pack_n - (int)group * d.pack, count = left < d.pack ? left : d.pack;
        if (count > 0) {
            if (r == count * full) return TileAt{(int)full, seg, count};
            if (r < count * full) return TileAt{(int)(r % full), seg + (int)(r / full), 1};
        }
        t -= d.pack_n * full + (d.pack_n + d.pack - 1) / d.pack;
        seg0 = d.pack_seg + d.pack_n;
    }
    // t / strips without a division, which every wavefront would wait for before
    // its first load: the quotient, or one more
    unsigned q = d.strips_inv == 0 ? t : (unsigned)((unsigned long long)t * d.strips_inv >> 32);
    if (q * strips > t) --q;
    return TileAt{(int)(t - q * strips), (int)(seg0 + q), 1};
}

// The tiles of `ty` rows of a descriptor, narrow last strips packed or not.
inline void set_tiles(GridDesc& d, int ty, bool pack) {
    d.ty = ty;
    d.nstrips = (d.nx + OWN - 1) / OWN;
    d.nsegs = (d.ny + ty - 1) / ty;
    d.strips_inv = d.nstrips == 1 ? 0 : (unsigned)(((1ull << 32) + d.nstrips - 1) / d.nstrips);
    int lo, hi;
    tile_range(d.nx, OWN, d.nstrips, d.nstrips - 1, lo, hi);
    d.pack = pack ? WAVE / (hi - lo + 2 * HALO) : 1;
    d.pack_seg = (HALO + ty - 1) / ty;
    d.pack_n = (d.ny - HALO) / ty - d.pack_seg;
    if (d.pack_n < 2 || d.pack < 2) { d.pack = 1; d.pack_n = 0; }
    d.ntiles = d.nstrips * d.nsegs - d.pack_n + (d.pack_n + d.pack - 1) / d.pack;
}

// Gives d the tiles of another descriptor of the grid.
inline void copy_tiles(GridDesc& d, const GridDesc& of) {
    d.ty = of.ty; d.nstrips = of.nstrips; d.nsegs = of.nsegs; d.ntiles = of.ntiles;
    d.strips_inv = of.strips_inv;
    d.pack = of.pack; d.pack_seg = of.pack_seg; d.pack_n = of.pack_n;
}

// Lane `lane` of tile w, whose columns are [x0, x1).
template <bool EDGE>
__host__ __device__ __forceinline__ TileLane tile_lane(const GridDesc& d, const TileAt& w, int x0, int x1, int lane) {
    int i = lane, k = 0;
    if (EDGE && w.count > 1) {
        const int span = x1 - x0 + 2 * HALO;
        k = lane / span;
        i = lane - k * span;
    }
    TileLane l;
    l.c = x0 - HALO + i;
    l.own = i >= HALO && l.c < x1 && k < w.count;
    l.use_x = i >= HALO - 1 && l.c < x1 && k < w.count;
    const LaneSource src = lane_source<EDGE>(d, l.c);
    l.side = src.side;
    l.row = EDGE ? (k < w.count ? k : w.count - 1) * d.ty : 0;
    l.at = src.c + l.row * d.pitch;
    return l;
}

template <bool EDGE>
__device__ __forceinline__ FirstRows first_rows(const GridDesc& d, const StageCtx& s, const TileLane& l, int j0) {
    FirstRows f;
#pragma unroll
    for (int q = 0; q < 4; ++q) f.r[q] = row_source<EDGE>(d, s, l, j0 - 2 + q);
    return f;
}

// apply_sponge (rki_kernel_sponge.F90:16-88) on one interior cell (c, j),
// 0-based: the distance to the nearest BC_SPONGE edge closer than the
// width sets alpha = strength ((width - d) / width)^2.  dsum collects the
// change of h.
__device__ __forceinline__ void sponge_cell(const GridDesc& d, double dt, int c, int j, double& h,
                                            double& hu, double& hv, double& dsum) {
    const int sw = d.sponge_width;
    int dmin = sw + 1;
    const int dw = c, de = d.nx - 1 - c, ds = j, dn = d.ny - 1 - j;
    if (d.bc[0] == BC_SPONGE && dw < sw && dw < dmin) dmin = dw;
    if (d.bc[1] == BC_SPONGE && de < sw && de < dmin) dmin = de;
    if (d.bc[2] == BC_SPONGE && ds < sw && ds < dmin) dmin = ds;
    if (d.bc[3] == BC_SPONGE && dn < sw && dn < dmin) dmin = dn;
    if (dmin < sw) {
        const double ratio = (double)(sw - dmin) / (double)sw;
        const double alpha = d.sponge_strength * ratio * ratio;
        const double h_in = h;
        h = h - dt * alpha * (h - d.sponge_h_ref);
        hu = hu - dt * alpha * hu;
        hv = hv - dt * alpha * hv;
        dsum = dsum + (h - h_in);
    }
}

// One tile of one RK stage: a strip of at most 60 owned columns x d.ty rows
// (or several such segments of a narrow strip), processed by one wavefront
// marching down the rows; lane l holds column x0 - 2 + l, so the two columns
// each side that the stencil needs are lanes of the same wavefront, and no
// column is treated apart.
// Row j: the y-slope of row j+1 is formed from the raw rows j, j+1, j+2
// held in registers, giving the face above row j together with the top
// state of row j carried from the previous row; the march starts one row
// early for the face below the first row.  The x-slope of row j takes the
// neighbours' differences by wave shuffles, each lane evaluates the face on
// its right and takes the face on its left from the lane before it.
//
// Bound by instruction issue: 60 of 64 lanes own a column (6 % of the work
// is halo).  The former layout, 64 owned columns with the edge columns
// batched one row per lane into LDS, spent 18 % of a 16-row tile in its
// prologue (plain divisions, 4096^2) and read 34 selects a row from LDS.
//
// A row whose stencil holds a non-zero value outside [2^-300, 2^40] in
// magnitude, or a non-finite one (unbounded()), anywhere in the wavefront is
// evaluated with plain divisions and the branches of the reference; every
// other row on the row path of swe_core.hpp.  Both give the same bits where
// both apply.
// STAGE 1 writes U* to B; STAGE 2 reads U* and U^n, applies the RK2 average
// and writes U^{n+1} over A, returning the lane's max CFL speed.
template <int STAGE, bool HLLC, bool EDGE, bool NF, bool REC, int FEAT = 0>
__device__ __forceinline__ double process_tile(const GridDesc& d, const StageCtx& s, TileRing& ring,
                                               const TileLane& l, const FirstRows& first, int j0, int j1, double& fsum,
                                               double& ssum) {
    constexpr bool FRC = (FEAT & FEAT_FORCING) != 0;
    constexpr bool SPG = (FEAT & FEAT_SPONGE) != 0;
    const int lane = threadIdx.x;
    const bool own = l.own, use_x = l.use_x;
    const double g = d.g;
    const long long pitch = d.pitch;
    // the row path's ranges assume a gravity and a friction of ordinary size
    const bool plain = d.plain_rows || !(g >= 1.0e-3 && g <= 1.0e6) ||
                       (!NF && s.src.has_friction && !(g * s.src.n_sq >= 0x1p-600));
    CflMax smax{0.0, 0.0};
    const bool same = d.dx == d.dy;
    const bool two_op = d.sdx.two_op && d.sdy.two_op;
    double facc = 0.0;  // sum of the lane's flux_h, rows in order
    double sacc = 0.0;  // sum of the lane's sponge change of h
    const bool read_un = STAGE == 2 || (STAGE == 3 && s.blend);

    // the rows j, j+1 and j+2 of the march, in LDS; a lane's neighbours by
    // their lane, the wavefront's ends repeating themselves (unused)
    const int lane_m = max(lane - 1, 0), lane_p = min(lane + 1, WAVE - 1);
    auto surf = [&](int slot, int i) { return Surf{ring.v[slot][0][i], ring.v[slot][1][i], ring.v[slot][2][i]}; };
    auto cell = [&](int slot, int i) {
        return Cell{ring.v[slot][4][i], ring.v[slot][1][i], ring.v[slot][2][i], ring.v[slot][3][i]};
    };
    auto put = [&](int slot, const Cell& x) {
        ring.v[slot][0][lane] = x.h + x.b; ring.v[slot][1][lane] = x.hu; ring.v[slot][2][lane] = x.hv;
        ring.v[slot][3][lane] = x.b; ring.v[slot][4][lane] = x.h;
    };
    auto hand_up = [&](const FState& hi, const Face& f, const Surf& dm) {
        ring.up[0][lane] = hi.h; ring.up[1][lane] = hi.hu; ring.up[2][lane] = hi.hv;
        ring.up[3][lane] = f.fh; ring.up[4][lane] = f.fhu; ring.up[5][lane] = f.fhv; ring.up[6][lane] = f.a;
        ring.up[7][lane] = dm.e; ring.up[8][lane] = dm.hu; ring.up[9][lane] = dm.hv;
    };
    // per row of the ring, over the wavefront: a value out of the row path's
    // bounds; the lanes below the dry tolerance; those in a thin layer
    struct RowBits {
        bool odd;
        unsigned long long dry, thin;
    };
    auto bits = [&](const Cell& x) {
        return RowBits{(bool)__any(unbounded(x)), __ballot(x.h < DRY_TOLERANCE), __ballot(x.h < THIN_LAYER_THRESHOLD)};
    };
    int sc = 0, sn = 1, snn = 2;
    bool odd_prev;
    RowBits bc, bn, bnn;
    {
        const Cell a = row_cell<EDGE, FEAT>(d, s, l, j0 - 2, first.r[0]);
        const Cell rc = row_cell<EDGE, FEAT>(d, s, l, j0 - 1, first.r[1]);
        const Cell rn = row_cell<EDGE, FEAT>(d, s, l, j0, first.r[2]);
        const Cell rnn = row_cell<EDGE, FEAT>(d, s, l, j0 + 1, first.r[3]);
        FState lo, hi;
        cell_states(a, rc, rn, lo, hi);
        odd_prev = __any(unbounded(a));
        bc = bits(rc);
        bn = bits(rn);
        bnn = bits(rnn);
        put(0, rc);
        put(1, rn);
        put(2, rnn);
        wave_lds_order();
        hand_up(hi, Face{0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, surf(1, lane) - surf(0, lane));
    }

    for (int j = j0 - 1; j < j1; ++j) {
        const bool inner = j >= j0;   // the row before the first only gives its upper face
        const bool plain_row = plain || odd_prev || bc.odd || bn.odd || bnn.odd;
        double fh = 0.0, fhu = 0.0, fhv = 0.0;   // the row's flux divergence
        auto faces = [&](auto exact) {
            constexpr bool EX = decltype(exact)::value;
            // y: slope of row j+1 and the face between rows j and j+1
            YPart y;
            {
                const FState tc{ring.up[0][lane], ring.up[1][lane], ring.up[2][lane]};
                const double b_c = ring.v[sc][3][lane], b_n = ring.v[sn][3][lane];
                const Surf n = surf(sn, lane), dp = surf(snn, lane) - n;
                FState lo, tn;
                Face fyt;
                if (EX) {
                    cell_states(cell(sc, lane), cell(sn, lane), cell(snn, lane), lo, tn);
                    fyt = face_flux<HLLC, true>(g, tc, b_c, lo, b_n);
                } else {
                    const Surf dm{ring.up[7][lane], ring.up[8][lane], ring.up[9][lane]};
                    states_row(dm, dp, n, b_n, __builtin_amdgcn_inverse_ballot_w64(bn.thin | bc.dry | bnn.dry), lo,
                               tn);
                    fyt = face_row<HLLC, true>(g, tc, b_c, lo, b_n, own);
                }
                const Face fyb{ring.up[3][lane], ring.up[4][lane], ring.up[5][lane], ring.up[6][lane], 0.0, 0.0};
                if (EX) y = divergence_y<DIV_PLAIN>(g, d.sdy, fyb, fyt);
                else if (two_op) y = divergence_y<DIV_TWO_OP>(g, d.sdy, fyb, fyt);
                else y = divergence_y<DIV_SHARED>(g, d.sdy, fyb, fyt);
                hand_up(tn, fyt, dp);
            }
            if (!inner) return;

            // x: slope of row j, the face right of each cell, the face left of it from the lane before
            const double b_c = ring.v[sc][3][lane], b_p = ring.v[sc][3][lane_p];
            FState lo, hi;
            Face fxl, fxr;
            if (EX) {
                cell_states(cell(sc, lane_m), cell(sc, lane), cell(sc, lane_p), lo, hi);
                fxr = face_flux<HLLC, false>(g, hi, b_c, shfl_down1(lo), b_p);
            } else {
                const Surf q = surf(sc, lane);
                states_row(q - surf(sc, lane_m), surf(sc, lane_p) - q, q, b_c,
                           __builtin_amdgcn_inverse_ballot_w64(bc.thin | (bc.dry << 1) | (bc.dry >> 1)), lo, hi);
                fxr = face_row<HLLC, false>(g, hi, b_c, shfl_down1(lo), b_p, use_x);
            }
            fxl.fh = shfl_up1(fxr.fh); fxl.fhu = shfl_up1(fxr.fhu); fxl.fhv = shfl_up1(fxr.fhv);
            fxl.a = shfl_up1(fxr.a);
            fxl.c = 0.0; fxl.d = 0.0;
            if (EX) divergence<DIV_PLAIN>(g, d.sdx, fxl, fxr, y, fh, fhu, fhv);
            else if (two_op) divergence<DIV_TWO_OP>(g, d.sdx, fxl, fxr, y, fh, fhu, fhv);
            else divergence<DIV_SHARED>(g, d.sdx, fxl, fxr, y, fh, fhu, fhv);
        };
        // Row j+3, needed at the end of the row, before the faces (4096^2, three
        // grids: 937 us a step, 948 with the loads after them; its eight registers
        // fit without spills).  The loads are unconditional (the last row of the
        // halo again, a cell of the grid): under a condition the compiler waits
        // for everything in flight where the paths join.
        const int jn = min(j + 3, j1 + 1);
        const Cell src = row_source<EDGE>(d, s, l, jn);
        __builtin_amdgcn_sched_barrier(0);
        if (__builtin_expect(plain_row, 0)) faces(ExactTag<true>{});
        else faces(ExactTag<false>{});

        // U^n of the cell (lanes that own none load their source cell's): the cell
        // update hides it, and the faces keep their registers
        Cell un{0.0, 0.0, 0.0, 0.0};
        if (read_un) {
            const long long k = (long long)max(j, 0) * pitch + l.at;
            un.h = in_hbm(d.ah)[k]; un.hu = in_hbm(d.ahu)[k]; un.hv = in_hbm(d.ahv)[k];
        }

        double h = 0.0, hu = 0.0, hv = 0.0;   // the row's result
        if (inner && own) {
            const long long k = (long long)j * pitch + l.at;
            if (REC) {
                in_hbm(d.rec)[k] = fh; in_hbm(d.rec)[d.plane + k] = fhu; in_hbm(d.rec)[2 * d.plane + k] = fhv;
            }
            Frc fr{0.0, 0.0, 0.0, 0.0, 0.0};
            if (FRC) {
                fr.wx = in_hbm(d.fwx)[k];
                fr.wy = in_hbm(d.fwy)[k];
                fr.dpdx = in_hbm(d.fdpx)[k];
                fr.dpdy = in_hbm(d.fdpy)[k];
                fr.rain = in_hbm(d.frain)[k];
            }
            const double n_cell = NF ? in_hbm(d.nfield)[k] : 0.0;
            double relax = 0.0;
            // the cell update; true where it has to be redone with plain divisions
            auto update = [&](auto exact) -> bool {
                constexpr bool EX = decltype(exact)::value;
                relax = 0.0;
                h = ring.v[sc][4][lane]; hu = ring.v[sc][1][lane]; hv = ring.v[sc][2][lane];
                if (EX) stage_body<NF, FRC>(s.src, s.dt, fh, fhu, fhv, h, hu, hv, n_cell, fr);
                else if (stage_body_row<NF, FRC>(s.src, s.dt, fh, fhu, fhv, h, hu, hv, n_cell, fr)) return true;
                // the sponge follows each fused stage (rki_solver.F90:787,814)
                if (STAGE == 1 && SPG) sponge_cell(d, s.dt, l.c, j + l.row, h, hu, hv, relax);
                if (STAGE == 2) {
                    // rki_kernel_fused.F90:435-463
                    h = 0.5 * (un.h + h);
                    hu = 0.5 * (un.hu + hu);
                    hv = 0.5 * (un.hv + hv);
                }
                if (STAGE == 3 && s.blend) {  // compute_ssp_combine, rki_kernel_update.F90:183-206
                    h = s.alpha * un.h + s.a_prev * h;
                    hu = s.alpha * un.hu + s.a_prev * hu;
                    hv = s.alpha * un.hv + s.a_prev * hv;
                }
                if (STAGE == 2 || (STAGE == 3 && s.blend)) {
                    if (EX) clamp_desing(g, h, hu, hv);
                    else if (clamp_row(g, h, hu, hv)) return true;
                }
                // :919-920, at beta_i dt in the generic schemes
                if (STAGE != 1 && SPG) sponge_cell(d, s.dt, l.c, j + l.row, h, hu, hv, relax);
                if (STAGE == 2 || (STAGE == 3 && s.last)) {
                    if (EX) cfl_plain(g, h, hu, hv, smax);
                    else cfl_row(g, same, h, hu, hv, smax);
                }
                return false;
            };
            if (__builtin_expect(plain_row, 0) || __builtin_expect(update(ExactTag<false>{}), 0))
                update(ExactTag<true>{});
            facc = facc + fh;
            sacc = sacc + relax;
        }

        // The prefetched row is waited for before the stores are issued:
        // loads and stores share one in-order counter, and a wait after the
        // stores waits for them too (a quarter of a row's time, 4096^2).
        Cell nxt{0.0, 0.0, 0.0, 0.0};
        odd_prev = bc.odd;
        bc = bn;
        bn = bnn;
        if (j + 1 < j1) {
            nxt = row_cell<EDGE, FEAT>(d, s, l, jn, src);
            bnn = bits(nxt);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (inner && own) {
            const long long k = (long long)j * pitch + l.at;
            if ((STAGE == 1 || (STAGE == 3 && s.first)) && d.sh != nullptr) {
                // h0, hu0, hv0 (rki_kernel_fused.F90:224-226, rki_solver.F90:879-881)
                in_hbm(d.sh)[k] = ring.v[sc][4][lane]; in_hbm(d.shu)[k] = ring.v[sc][1][lane]; in_hbm(d.shv)[k] = ring.v[sc][2][lane];
            }
            in_hbm(s.oh)[k] = h; in_hbm(s.ohu)[k] = hu; in_hbm(s.ohv)[k] = hv;
        }
        wave_lds_order();
        put(sc, nxt);   // row j+3 takes the place of row j
        wave_lds_order();
        const int free_slot = sc;
        sc = sn; sn = snn; snn = free_slot;
    }
    fsum = facc;
    ssum = sacc;
    return cfl_max(smax, same, d.dx, d.dy);
}

}  // namespace rk
