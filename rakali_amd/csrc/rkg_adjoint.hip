// rkg_adjoint.hip -- discrete adjoint of the SSP-RK2 step: gradients of a
// gauge sea-surface misfit with respect to the bed, the per-cell Manning n
// and the initial state.
//
// Loss: L = sum over steps s and gauges k of (eta_k(t_s) - target_{s,k})^2,
// eta = h + b at the gauge cell after step s.  The forward pass runs the
// ordinary stage kernels (per-cell Manning n) and keeps the state every
// `checkpoint_interval` steps.  The reverse sweep takes segments last to
// first: it replays a segment from its checkpoint with the recording stage
// kernels, which keep U^n, U* and each stage's flux divergence for every
// step of the segment, then reverses the steps one by one:
//   k_adj_body  -- cell-local: RK2 average, clamp, KP07, Froude backstop,
//                  Manning and Coriolis transposed; emits the adjoint of the
//                  flux divergence of every cell and the Manning gradient;
//   k_adj_y     -- tile kernel, rows marched: every y face and y slope of
//                  the stage, with the south / north ghost rows;
//   k_adj_x     -- row-local: every x face and x slope, with the west /
//                  east ghost columns; both add onto the adjoint of the
//                  stage input and the bed.
//   k_dt_rev    -- one workgroup per step: the dependence of the loss on the
//                  step's dt (update, friction, Coriolis angle, the tide's
//                  clock t_{s+1} = t_s + dt_s) and, for a CFL dt, on the
//                  cell that set the max speed (k_adj_body<1> finds it).
// The gradient is that of the discrete scheme with its dt rule: fixed dt,
// the CFL dt every cfl_interval steps, and the t_end bound.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "../../include/rakali_amd.h"
#include "adjoint.hpp"
#include "gauge_eval.hpp"
#include "rkg_internal.hpp"
#include "stage_kernels.hpp"

using namespace rk;

namespace {

constexpr unsigned ADJ_MAGIC = 0x72616B41u;  // 'rakA'
constexpr unsigned ADJ_DEAD = 0xDEADBEEFu;
constexpr int AW = 60;                        // own columns per workgroup of k_adj_x

struct AdjStage {
    GridDesc d;                 // geometry, physics, bed, n field; ah.. = stage input V
    const double* un;           // U^n (3 planes), stage 2
    const double* div;          // recorded flux divergence (3 planes)
    double* lam_in;             // adjoint of the stage input (3 planes)
    double* lam_out;            // adjoint of the stage output (3 planes); stage 2: the
                                // adjoint of U^{n+1} in, replaced by its U^n part
    double* lam_div;            // 3 planes
    double* grad_b;
    double* grad_n;
    const double* hist;         // (t, dt, dt recomputed) of the step
    double* part_dt;            // per body workgroup: sum of d L / d dt of its cells
    double* pval;               // stage 1 with the CFL dt: per body workgroup, max CFL speed of
    long long* pidx;            // the stage input and its first cell (x fastest), else null
    double* edge_eta;           // d L / d eta through every tidal ghost cell, see edge_slot
    int edge_len;               // max(nx, ny)
    int ty;                     // rows per tile of k_adj_y
};

// Slot of ghost layer kk (0 = next to the edge) at position p along edge e
// (0 W, 1 E, 2 S, 3 N) in edge_eta.
__host__ __device__ __forceinline__ long long edge_slot(int e, int kk, int p, int len) {
    return (long long)(e * 2 + kk) * len + p;
}

constexpr int HIST = 3;         // doubles per step in hist

__device__ __forceinline__ SourceTerms adj_src(const GridDesc& d, double dt) {
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

// Sum over a 256-thread workgroup in a fixed order; the result is valid in
// thread 0.
__device__ __forceinline__ double block_sum256(double v, double* red4) {
    v = wave_sum(v);
    if ((threadIdx.x & (WAVE - 1)) == 0) red4[threadIdx.x / WAVE] = v;
    __syncthreads();
    double r = 0.0;
    if (threadIdx.x == 0) r = ((red4[0] + red4[1]) + red4[2]) + red4[3];
    __syncthreads();
    return r;
}

// Cell-local reverse of one stage.  STAGE 2: lam_out holds the adjoint of
// U^{n+1} and is replaced by the U^n part of the RK2 average; lam_in (the
// adjoint of U*) is written.  STAGE 1: lam_out is the adjoint of U* and
// lam_in (the adjoint of U^n) is added to.
template <int STAGE>
__device__ __forceinline__ void adj_body(const AdjStage& a, int blk, int nblk) {
    const GridDesc& d = a.d;
    const double dt = a.hist[1];
    const SourceTerms src = adj_src(d, dt);
    const long long P = d.plane;
    const long long n = (long long)d.nx * d.ny;
    double ldt = 0.0;
    double best = 0.0;   // stage 1: max CFL speed of U_s and its first cell
    long long bi = -1;
    for (long long idx = blk * 256ll + threadIdx.x; idx < n; idx += (long long)nblk * 256) {
        const int j = (int)(idx / d.nx), i = (int)(idx % d.nx);
        const long long k = (long long)j * d.pitch + i;
        const double v0 = d.ah[k], v1 = d.ahu[k], v2 = d.ahv[k];
        if (STAGE == 1 && a.pval) {
            const double sp = adj::cfl_speed_fwd(d.g, d.dx, d.dy, v0, v1, v2);
            if (sp > best) { best = sp; bi = idx; }
        }
        const adj::S3 div{a.div[k], a.div[P + k], a.div[2 * P + k]};
        const double nc = d.nfield ? d.nfield[k] : d.manning_n;
        const double nsq = d.nfield ? nc * nc : src.n_sq;
        const bool fr = d.nfield ? (nc > 0.0) : (src.has_friction != 0);
        adj::S3 lw;
        if (STAGE == 2) {
            double wh = v0, whu = v1, whv = v2;
            adj::body_fwd(src, dt, div, nsq, fr, wh, whu, whv);
            const double ah = 0.5 * (a.un[k] + wh), ahu = 0.5 * (a.un[P + k] + whu), ahv = 0.5 * (a.un[2 * P + k] + whv);
            const adj::S3 lo{a.lam_out[k], a.lam_out[P + k], a.lam_out[2 * P + k]};
            const adj::S3 la = adj::clamp_rev(d.g, ah, ahu, ahv, lo);
            lw = adj::S3{0.5 * la.h, 0.5 * la.hu, 0.5 * la.hv};
            a.lam_out[k] = lw.h; a.lam_out[P + k] = lw.hu; a.lam_out[2 * P + k] = lw.hv;
        } else {
            lw = adj::S3{a.lam_out[k], a.lam_out[P + k], a.lam_out[2 * P + k]};
        }
        const adj::BodyRev r = adj::body_rev(src, dt, div, nc, nsq, fr, v0, v1, v2, lw);
        if (STAGE == 2) {
            a.lam_in[k] = r.lv.h; a.lam_in[P + k] = r.lv.hu; a.lam_in[2 * P + k] = r.lv.hv;
        } else {
            a.lam_in[k] += r.lv.h; a.lam_in[P + k] += r.lv.hu; a.lam_in[2 * P + k] += r.lv.hv;
        }
        a.lam_div[k] = r.ldiv.h; a.lam_div[P + k] = r.ldiv.hu; a.lam_div[2 * P + k] = r.ldiv.hv;
        if (d.nfield && a.grad_n) a.grad_n[k] += r.ln;
        ldt = ldt + r.ldt;
    }
    __shared__ double red4[4];
    const double tot = block_sum256(ldt, red4);
    if (threadIdx.x == 0) a.part_dt[blk] = tot;
    if (STAGE == 1 && a.pval) {
        __shared__ double sv[256];
        __shared__ long long si[256];
        sv[threadIdx.x] = best;
        si[threadIdx.x] = bi;
        __syncthreads();
        for (int s = 128; s > 0; s >>= 1) {
            if (threadIdx.x < s) {
                const double v = sv[threadIdx.x + s];
                const long long x = si[threadIdx.x + s];
                if (v > sv[threadIdx.x] || (v == sv[threadIdx.x] && x >= 0 && (si[threadIdx.x] < 0 || x < si[threadIdx.x]))) {
                    sv[threadIdx.x] = v;
                    si[threadIdx.x] = x;
                }
            }
            __syncthreads();
        }
        if (threadIdx.x == 0) { a.pval[blk] = sv[0]; a.pidx[blk] = si[0]; }
    }
}

template <int STAGE>
__global__ __launch_bounds__(256) void k_adj_body(AdjStage a) {
    adj_body<STAGE>(a, blockIdx.x, gridDim.x);
}

struct Acc {   // adjoint accumulator of one cell: (h, hu, hv, b)
    double h, hu, hv, b;
};

__device__ __forceinline__ void add(Acc& a, const adj::C4& c) { a.h += c.h; a.hu += c.hu; a.hv += c.hv; a.b += c.b; }
__device__ __forceinline__ adj::C4 c4(const Acc& a) { return adj::C4{a.h, a.hu, a.hv, a.b}; }
__device__ __forceinline__ double sh_dn(double v) { return __shfl_down(v, 1, WAVE); }
__device__ __forceinline__ double sh_up(double v) { return __shfl_up(v, 1, WAVE); }
__device__ __forceinline__ adj::C4 sh_dn(const adj::C4& c) { return adj::C4{sh_dn(c.h), sh_dn(c.hu), sh_dn(c.hv), sh_dn(c.b)}; }
__device__ __forceinline__ adj::C4 sh_up(const adj::C4& c) { return adj::C4{sh_up(c.h), sh_up(c.hu), sh_up(c.hv), sh_up(c.b)}; }
__device__ __forceinline__ adj::C4 sh_from(const adj::C4& c, int src) {
    return adj::C4{__shfl(c.h, src, WAVE), __shfl(c.hu, src, WAVE), __shfl(c.hv, src, WAVE), __shfl(c.b, src, WAVE)};
}

// The planes a row of a face reverse needs, in the order of the LDS rows: the
// stage input (h, hu, hv, b), the adjoint of the flux divergence, and what the
// row adds to, the adjoint of the input and the bed gradient.
constexpr int ADJ_PLANES = 11;

__device__ __forceinline__ const double* adj_plane(const AdjStage& a, int p) {
    const GridDesc& d = a.d;
    if (p < 3) return d.ah + p * d.plane;   // ah, ahu, ahv follow each other
    if (p == 3) return d.bed;
    if (p < 7) return a.lam_div + (p - 4) * d.plane;
    if (p < 10) return a.lam_in + (p - 7) * d.plane;
    return a.grad_b;
}

// 16 bytes per lane from memory into 64 x 16 bytes of LDS, without registers.
__device__ __forceinline__ void to_lds(const double* src, double* dst) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

// Waits for every load of the wavefront before what follows (the stores of a
// row, which share the loads' in-order counter: a row's loads must not be
// waited for behind the stores of the row before).
__device__ __forceinline__ void wait_loads() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
}

// A ghost cell of side `side` from its source cell (see lane_source).
__device__ __forceinline__ Cell side_ghost(const GridDesc& d, int side, double eta, const Cell& src) {
    return ghost_from(d, d.bc[side], eta, src, src, (side & 1) ? 1.0 : -1.0, side < 2);
}

// Adjoint of the row-y ghost at column x onto interior cells (x-direction
// ghosts: normal momentum hu); cell(col) gives the row's interior cells.
// Returns the contributions for the mirror and first-interior columns, and in
// leta that for the tide.
template <class CELL>
__device__ __forceinline__ void ghost_x_rev(const GridDesc& d, double eta, int x, CELL cell, const adj::C4& lg, int& mcol,
                                            int& icol, adj::C4& lm, adj::C4& li, double* leta) {
    const bool west = x < 0;
    const int kk = west ? (-x - 1) : (x - d.nx);
    mcol = west ? kk : (d.nx - 1 - kk);
    icol = west ? 0 : (d.nx - 1);
    lm = adj::C4{0, 0, 0, 0};
    li = adj::C4{0, 0, 0, 0};
    adj::ghost_rev(d.bc[west ? 0 : 1], d.g, eta, d.inflow_velocity, d.clamped_elevation, cell(mcol), cell(icol),
                   west ? -1.0 : 1.0, true, lg, lm, li, leta);
}

__device__ __forceinline__ void ghost_y_rev(const GridDesc& d, double eta, bool south, const Cell& mir, const Cell& in0,
                                            const adj::C4& lg, adj::C4& lm, adj::C4& li, double* leta) {
    lm = adj::C4{0, 0, 0, 0};
    li = adj::C4{0, 0, 0, 0};
    adj::ghost_rev(d.bc[south ? 2 : 3], d.g, eta, d.inflow_velocity, d.clamped_elevation, mir, in0,
                   south ? -1.0 : 1.0, false, lg, lm, li, leta);
}

// Two LDS rows of the 11 planes over 64 columns (the twelfth is a spare: two
// planes make one load), and what waits for ghost rows: the south ghost rows'
// accumulators, then row ny-2's old values, accumulator and cell.
struct YRows {
    double v[2][ADJ_PLANES + 1][WAVE];
    double kept[12][WAVE];
};

// Reverse of the y faces and y slopes of one stage (and the south / north
// ghost rows) onto the stage input and the bed.  One wavefront per tile of
// 64 whole columns (lane l holds column c0 + l; this direction is
// column-local, so no halo columns) and rows [j0, j1).  The rows are
// marched from j0 - 2 to j1: iteration r reverses the y face between rows
// r and r+1 and the y slope of row r, which completes row r-1.  A ghost row's
// adjoint is added to its source rows when row 0 is complete (south), or with
// the last row (north, row ny-2 waiting for it).  TY: a south or north edge is
// tidal, and what its ghost cells give the tide is kept in edge_eta for
// k_dt_rev.
//
// Bound by latency with two wavefronts on a SIMD (face_rev's live values leave
// no room for a third): what iteration r + 1 needs is loaded into LDS during
// iteration r, so that a row waits for no memory.  1024^2:
// 57 us when each row loaded its own, 48 now, of which its 126 MB take 27.
template <bool HLLC, int STAGE, bool TY>
__device__ __forceinline__ void adj_y(const AdjStage& a, YRows& rows, int blk) {
    const GridDesc& d = a.d;
    const int lane = threadIdx.x;
    const int nstr = (d.nx + WAVE - 1) / WAVE;
    const int sx = blk % nstr, sy = blk / nstr;
    const int c0 = sx * WAVE;
    int j0, j1;
    tile_range(d.ny, a.ty, (d.ny + a.ty - 1) / a.ty, sy, j0, j1);
    const int x = c0 + lane;
    const bool xin = x < d.nx;   // lanes past the edge compute on the rows' padding, unwritten
    const int xs = xin ? x : d.nx - 1;
    const bool south = j0 < 3, north = j1 + 2 >= d.ny;
    const int ny = d.ny;
    const long long P = d.plane;

    // lane l loads columns 2 (l % 32) and the next of planes 2 i and 2 i + 1
    const int col = min(c0 + 2 * (lane & 31), (int)d.pitch - 2);
    const double* src[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) src[i] = adj_plane(a, min(2 * i + (lane >> 5), ADJ_PLANES - 1)) + col;
    // the source row of row j (lane_source's rule for rows)
    auto source_row = [&](int j) {
        if (j < 0) return min(mirrors(d.bc[2]) ? -j - 1 : 0, ny - 1);
        if (j >= ny) return max(mirrors(d.bc[3]) ? 2 * ny - 1 - j : ny - 1, 0);
        return j;
    };
    auto fetch = [&](int r, int buf) {   // what iteration r needs
        const long long ov = source_row(r + 2) * d.pitch, od = min(max(r + 1, 0), ny - 1) * d.pitch,
                        ol = min(max(r - 1, 0), ny - 1) * d.pitch;
        const long long o67 = lane < WAVE / 2 ? od : ol;
        to_lds(src[0] + ov, rows.v[buf][0]);
        to_lds(src[1] + ov, rows.v[buf][2]);
        to_lds(src[2] + od, rows.v[buf][4]);
        to_lds(src[3] + o67, rows.v[buf][6]);
        to_lds(src[4] + ol, rows.v[buf][8]);
        to_lds(src[5] + ol, rows.v[buf][10]);
    };
    const int rs = j0 - 2, re = j1;
    const long long q0 = source_row(rs - 1) * d.pitch + xs, q1 = source_row(rs) * d.pitch + xs,
                    q2 = source_row(rs + 1) * d.pitch + xs;
    Cell v0{d.ah[q0], d.ahu[q0], d.ahv[q0], d.bed[q0]}, v1{d.ah[q1], d.ahu[q1], d.ahv[q1], d.bed[q1]},
        v2{d.ah[q2], d.ahu[q2], d.ahv[q2], d.bed[q2]}, v3;
    adj::S3 ld_r{0.0, 0.0, 0.0};
    if (rs >= 0) {
        const long long o = rs * d.pitch + xs;
        ld_r = adj::S3{a.lam_div[o], a.lam_div[P + o], a.lam_div[2 * P + o]};
    }
    fetch(rs, 0);
    const double tau = STAGE == 1 ? a.hist[0] : a.hist[0] + a.hist[1];   // bc%time of the stage
    // the tide (a long dependent chain) only where a tidal edge's ghosts are read
    const bool tidal = (south && d.bc[2] == BC_TIDAL) || (north && d.bc[3] == BC_TIDAL);
    const double eta = tidal ? tidal_eta(d, tau) : 0.0;
    auto row_ghost = [&](int j, const Cell& c) {
        if (j >= 0 && j < ny) return c;
        if (j < -2 || j > ny + 1) return Cell{0.0, 0.0, 0.0, 0.0};
        return side_ghost(d, j < 0 ? 2 : 3, eta, c);
    };
    if (south || north) {
        v0 = row_ghost(rs - 1, v0);
        v1 = row_ghost(rs, v1);
        v2 = row_ghost(rs + 1, v2);
    }
    const double g = d.g;
    const bool fast = g >= 1.0e-3 && g <= 1.0e6;   // face_rev_fast's ranges assume an ordinary gravity
    const double rdy = 1.0 / d.dy;

    Acc acc[3];   // rows r-1, r, r+1
#pragma unroll
    for (int q = 0; q < 3; ++q) acc[q] = Acc{0.0, 0.0, 0.0, 0.0};
    FState hi_r, lo_tmp;
    adj::states_fwd(v0, v1, v2, lo_tmp, hi_r);
    adj::S3 llo_r{0.0, 0.0, 0.0};        // adjoint of the y lo-state of row r (from face r - 1/2)

    // Adjoint of ghost row rho onto its mirror row (cell mir) and the first
    // interior row (cell in0).
    auto fold = [&](int rho, const Acc& ghost, const Cell& mir, const Cell& in0, adj::C4& lm, adj::C4& li) {
        const adj::C4 lg = c4(ghost);
        double leta = 0.0;
        ghost_y_rev(d, eta, rho < 0, mir, in0, lg, lm, li, &leta);
        const int e = rho < 0 ? 2 : 3;
        if (TY && xin && d.bc[e] == BC_TIDAL)
            a.edge_eta[edge_slot(e, rho < 0 ? -rho - 1 : rho - ny, x, a.edge_len)] = leta;
    };

    wait_loads();   // the rows of the first iteration
    for (int r = rs; r <= re; ++r) {
        // v0..v2 are rows r-1 .. r+1
        const double(*in)[WAVE] = rows.v[(r - rs) & 1];
        v3 = Cell{in[0][lane], in[1][lane], in[2][lane], in[3][lane]};
        adj::S3 ld_r1{in[4][lane], in[5][lane], in[6][lane]};
        const adj::C4 old{in[7][lane], in[8][lane], in[9][lane], in[10][lane]};   // row r-1
        if (r < re) fetch(r + 1, (r + 1 - rs) & 1);
        if (south || north) {
            v3 = row_ghost(r + 2, v3);
            if (r + 1 < 0 || r + 1 >= ny) ld_r1 = adj::S3{0.0, 0.0, 0.0};
        }
        FState lo_r1, hi_r1;
        adj::states_fwd(v1, v2, v3, lo_r1, hi_r1);
        // y face r + 1/2 (faces -1/2 .. ny - 1/2)
        adj::S3 lhi_r{0.0, 0.0, 0.0}, llo_r1{0.0, 0.0, 0.0};
        if (r >= -1 && r <= ny - 1) {
            const Face lf = adj::face_seed<true>(g, rdy, ld_r, ld_r1);
            double lbL = 0.0, lbR = 0.0;
            if (!(fast && adj::face_rev_fast<HLLC, true>(g, hi_r, v1.b, lo_r1, v2.b, lf, lhi_r, lbL, llo_r1, lbR,
                                                          xin)))
                adj::face_rev<HLLC, true>(g, hi_r, v1.b, lo_r1, v2.b, lf, lhi_r, lbL, llo_r1, lbR);
            acc[1].b += lbL;
            acc[2].b += lbR;
        }
        // y slope of row r
        {
            adj::C4 lm{0, 0, 0, 0}, lc{0, 0, 0, 0}, lp{0, 0, 0, 0};
            adj::states_rev(v0, v1, v2, llo_r, lhi_r, lm, lc, lp);
            add(acc[0], lm);
            add(acc[1], lc);
            add(acc[2], lp);
        }
        auto keep = [&](int q, double h, double hu, double hv, double lb) {
            rows.kept[q][lane] = h; rows.kept[q + 1][lane] = hu; rows.kept[q + 2][lane] = hv; rows.kept[q + 3][lane] = lb;
        };
        auto kept = [&](int q) {
            return Acc{rows.kept[q][lane], rows.kept[q + 1][lane], rows.kept[q + 2][lane], rows.kept[q + 3][lane]};
        };
        adj::C4 lm, li;
        if (j0 == 0 && r <= 1) {
            if (r == -1 || r == 0) {   // row -2, -1 complete
                keep(4 * (r + 1), acc[0].h, acc[0].hu, acc[0].hv, acc[0].b);
            } else if (r == 1) {       // acc[0], acc[1] and v0, v1 are rows 0 and 1
                fold(-2, kept(0), v1, v0, lm, li);
                add(acc[1], lm);       // the mirror row is 1, the first row 0
                add(acc[0], li);
                fold(-1, kept(4), v0, v0, lm, li);
                add(acc[0], lm);
                add(acc[0], li);
            }
        }
        const int rho = r - 1;
        auto put = [&](int row, const adj::C4& from, const Acc& more) {
            const long long k = row * d.pitch + x;
            a.lam_in[k] = from.h + more.h;
            a.lam_in[P + k] = from.hu + more.hu;
            a.lam_in[2 * P + k] = from.hv + more.hv;
            a.grad_b[k] = from.b + more.b;
        };
        const bool waits = j1 == ny && rho == ny - 2 && rho >= j0;
        if (waits) {
            keep(0, old.h, old.hu, old.hv, old.b);
            keep(4, acc[0].h, acc[0].hu, acc[0].hv, acc[0].b);
            keep(8, v0.h, v0.hu, v0.hv, v0.b);
        }
        if (j1 == ny && r == ny) {   // acc[0..2] are rows ny-1, ny, ny+1, v0 is row ny-1
            Acc last = kept(4);      // row ny-2
            const Acc cell = kept(8);
            fold(ny, acc[1], v0, v0, lm, li);
            add(acc[0], lm);
            add(acc[0], li);
            fold(ny + 1, acc[2], Cell{cell.h, cell.hu, cell.hv, cell.b}, v0, lm, li);
            add(last, lm);
            add(acc[0], li);
            if (xin) put(ny - 2, c4(kept(0)), last);
        }
        wait_loads();
        if (xin && rho >= j0 && rho < j1 && !waits) put(rho, old, acc[0]);
        acc[0] = acc[1];
        acc[1] = acc[2];
        acc[2] = Acc{0.0, 0.0, 0.0, 0.0};
        v0 = v1; v1 = v2; v2 = v3;
        hi_r = hi_r1;
        llo_r = llo_r1;
        ld_r = ld_r1;
    }
}

template <bool HLLC, int STAGE, bool TY>
__global__ __launch_bounds__(WAVE) void k_adj_y(AdjStage a) {
    __shared__ alignas(16) YRows rows;
    adj_y<HLLC, STAGE, TY>(a, rows, blockIdx.x);
}

// Two LDS rows of the 11 planes over 68 columns, 34 pairs each: the 374 pairs
// of a row are loaded 64 at a time.
// Rows per workgroup of k_adj_x: with the loads a row ahead a workgroup costs
// little to start, and many short ones even out the edge strips (us: 1024^2
// 4 rows 54, 2 rows 53, 9 rows 58; 4096 x 1024 4 rows 144, 32 rows 206).
constexpr int XROWS = 4;
constexpr int XCOLS = 68;
constexpr int XLOADS = (ADJ_PLANES * XCOLS / 2 + WAVE - 1) / WAVE;
struct XRows {
    double v[2][XLOADS * WAVE * 2];
};

// Reverse of the x faces and x slopes of one stage (and the west / east
// ghost columns) onto the stage input and the bed.  This direction is
// row-local: every row is independent.  One wavefront per strip of at
// most 60 owned columns [c0, c1) and XROWS rows; lane l holds column
// c0 - 2 + l, so the faces and slopes that touch an owned cell are all in
// the wavefront (lanes 0 and 63 need one column more).  The face right of a
// cell is reversed by the cell's lane; neighbours' parts move by lane
// shuffles; ghost columns fold onto their source columns by lane permutes.
// TX: a west or east edge is tidal (see k_adj_y's TY).
//
// Bound by latency, as adj_y: the next row is loaded into LDS while a row is
// computed.  1024^2: 78 us when each row loaded its own, 44 now,
// of which its 138 MB take 30; 4096 x 1024: 144 us, at 3.8 TB/s.
template <bool HLLC, int STAGE, bool TX>
__device__ __forceinline__ void adj_x(const AdjStage& a, XRows& rows, int blk) {
    const GridDesc& d = a.d;
    const int lane = threadIdx.x;
    const int nstr = (d.nx + AW - 1) / AW, nrow = (d.ny + XROWS - 1) / XROWS;
    // the edge strips, whose ghost columns take longer, first (1024^2: 45 us, 49
    // in the order of the columns)
    int sx, sy;
    if (nstr < 3) { sx = blk % nstr; sy = blk / nstr; }
    else if (blk < 2 * nrow) { sx = blk & 1 ? nstr - 1 : 0; sy = blk >> 1; }
    else { const int q = blk - 2 * nrow; sx = 1 + q % (nstr - 2); sy = q / (nstr - 2); }
    int c0, c1;
    tile_range(d.nx, AW, nstr, sx, c0, c1);
    const int r0 = sy * XROWS, r1 = min(r0 + XROWS, d.ny);
    const int x = c0 - 2 + lane;
    const bool own_col = x >= c0 && x < c1;
    // columns c0 - 3 .. c0 + 62 are read
    const bool edge_tile = c0 < 3 || c0 + 62 >= d.nx;
    const long long P = d.plane;
    // The LDS rows start at the even column cb; pairs outside the rows are
    // read from their ends and not used.
    const int cb = (c0 - 3) & ~1;
    const double* src[XLOADS];
#pragma unroll
    for (int i = 0; i < XLOADS; ++i) {
        const int q = i * WAVE + lane;
        const int p = min(q / (XCOLS / 2), ADJ_PLANES - 1);
        const int col = cb + 2 * (q % (XCOLS / 2));
        src[i] = adj_plane(a, p) + min(max(col, 0), (int)d.pitch - 2);
    }
    auto fetch = [&](int r, int buf) {
        const long long o = r * d.pitch;
#pragma unroll
        for (int i = 0; i < XLOADS; ++i) to_lds(src[i] + o, rows.v[buf] + i * WAVE * 2);
    };
    if (r0 < r1) fetch(r0, 0);
    const double tau = STAGE == 1 ? a.hist[0] : a.hist[0] + a.hist[1];
    // the tide only where a tidal edge's ghosts are read
    const bool tidal = (c0 < 3 && d.bc[0] == BC_TIDAL) || (c0 + 62 >= d.nx && d.bc[1] == BC_TIDAL);
    const double eta = tidal ? tidal_eta(d, tau) : 0.0;
    const double g = d.g;
    const bool fast = g >= 1.0e-3 && g <= 1.0e6;
    const double rdx = 1.0 / d.dx;
    const LaneSource l1 = edge_tile ? lane_source<true>(d, x) : lane_source<false>(d, x);
    const LaneSource l2 = edge_tile ? lane_source<true>(d, lane == 0 ? x - 1 : x + 1) : l1;
    const int i1 = min(max(l1.c - cb, 0), XCOLS - 1), i2 = min(max(l2.c - cb, 0), XCOLS - 1);
    wait_loads();   // the first row
    for (int r = r0; r < r1; ++r) {
        const double* row = rows.v[(r - r0) & 1];
        auto cell_at = [&](int i) { return Cell{row[i], row[XCOLS + i], row[2 * XCOLS + i], row[3 * XCOLS + i]}; };
        Cell v1 = cell_at(i1), xm, xp;
        adj::S3 ld_r{row[4 * XCOLS + i1], row[5 * XCOLS + i1], row[6 * XCOLS + i1]};
        const adj::C4 old{row[7 * XCOLS + i1], row[8 * XCOLS + i1], row[9 * XCOLS + i1], row[10 * XCOLS + i1]};
        if (!edge_tile) {
            xm = cell_at(i1 - 1);
            xp = cell_at(i1 + 1);
        } else {
            Cell out = cell_at(i2);
            const Cell zero{0.0, 0.0, 0.0, 0.0};
            if (l1.side != -1) {
                v1 = l1.side < 0 ? zero : side_ghost(d, l1.side, eta, v1);
                ld_r = adj::S3{0.0, 0.0, 0.0};
            }
            if (l2.side != -1) out = l2.side < 0 ? zero : side_ghost(d, l2.side, eta, out);
            xm.h = sh_up(v1.h); xm.hu = sh_up(v1.hu); xm.hv = sh_up(v1.hv); xm.b = sh_up(v1.b);
            xp.h = sh_dn(v1.h); xp.hu = sh_dn(v1.hu); xp.hv = sh_dn(v1.hv); xp.b = sh_dn(v1.b);
            if (lane == 0) xm = out;
            if (lane == WAVE - 1) xp = out;
        }
        if (r + 1 < r1) fetch(r + 1, (r + 1 - r0) & 1);
        FState lo_x, hi_x;
        adj::states_fwd(xm, v1, xp, lo_x, hi_x);
        FState R;
        R.h = sh_dn(lo_x.h); R.hu = sh_dn(lo_x.hu); R.hv = sh_dn(lo_x.hv);
        const adj::S3 ld_next{sh_dn(ld_r.h), sh_dn(ld_r.hu), sh_dn(ld_r.hv)};
        adj::S3 lhi_x{0.0, 0.0, 0.0}, lR{0.0, 0.0, 0.0};
        double lbL = 0.0, lbR = 0.0;
        if (lane < WAVE - 1 && x >= -1 && x <= d.nx - 1) {   // the face between x and x + 1
            const Face lf = adj::face_seed<false>(g, rdx, ld_r, ld_next);
            if (!(fast && adj::face_rev_fast<HLLC, false>(g, hi_x, v1.b, R, xp.b, lf, lhi_x, lbL, lR, lbR, true)))
                adj::face_rev<HLLC, false>(g, hi_x, v1.b, R, xp.b, lf, lhi_x, lbL, lR, lbR);
        }
        adj::S3 llo_x{sh_up(lR.h), sh_up(lR.hu), sh_up(lR.hv)};
        const double lb_from_left = sh_up(lbR);
        if (lane == 0) llo_x = adj::S3{0.0, 0.0, 0.0};
        adj::C4 mine{0.0, 0.0, 0.0, lbL + (lane == 0 ? 0.0 : lb_from_left)};
        adj::C4 lm{0, 0, 0, 0}, lc{0, 0, 0, 0}, lp{0, 0, 0, 0};
        adj::states_rev(xm, v1, xp, llo_x, lhi_x, lm, lc, lp);
        const adj::C4 from_right = sh_dn(lm);   // lane l+1's left-neighbour part
        const adj::C4 from_left = sh_up(lp);    // lane l-1's right-neighbour part
        mine.h += lc.h; mine.hu += lc.hu; mine.hv += lc.hv; mine.b += lc.b;
        if (lane < WAVE - 1) { mine.h += from_right.h; mine.hu += from_right.hu; mine.hv += from_right.hv; mine.b += from_right.b; }
        if (lane > 0) { mine.h += from_left.h; mine.hu += from_left.hu; mine.hv += from_left.hv; mine.b += from_left.b; }
        // ghost columns fold onto their source columns (tiles at an edge only)
        if (edge_tile) {
            adj::C4 gm{0, 0, 0, 0}, gi{0, 0, 0, 0};
            int mcol = -100, icol = -100;
            if (x == -1 || x == -2 || x == d.nx || x == d.nx + 1) {
                double leta = 0.0;
                ghost_x_rev(d, eta, x, [&](int c) { return cell_at(c - cb); }, mine, mcol, icol, gm, gi, &leta);
                const int e = x < 0 ? 0 : 1;
                // kept once, by the tile holding the edge column
                if (TX && (x < 0 ? c0 == 0 : c1 == d.nx) && d.bc[e] == BC_TIDAL)
                    a.edge_eta[edge_slot(e, x < 0 ? -x - 1 : x - d.nx, r, a.edge_len)] = leta;
            }
            // lanes holding columns -2, -1, nx, nx + 1 (when inside the wavefront)
            const int srcs[4] = {-c0, 1 - c0, d.nx - c0 + 2, d.nx - c0 + 3};
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int src = srcs[s];
                if (src < 0 || src >= WAVE) continue;
                const adj::C4 rm = sh_from(gm, src), ri = sh_from(gi, src);
                const int rmcol = __shfl(mcol, src, WAVE), ricol = __shfl(icol, src, WAVE);
                if (x == rmcol) { mine.h += rm.h; mine.hu += rm.hu; mine.hv += rm.hv; mine.b += rm.b; }
                if (x == ricol) { mine.h += ri.h; mine.hu += ri.hu; mine.hv += ri.hv; mine.b += ri.b; }
            }
        }
        wait_loads();
        if (own_col) {
            const long long k = r * d.pitch + x;
            a.lam_in[k] = old.h + mine.h;
            a.lam_in[P + k] = old.hu + mine.hu;
            a.lam_in[2 * P + k] = old.hv + mine.hv;
            a.grad_b[k] = old.b + mine.b;
        }
    }
}

template <bool HLLC, int STAGE, bool TX>
__global__ __launch_bounds__(WAVE) void k_adj_x(AdjStage a) {
    __shared__ alignas(16) XRows rows;
    adj_x<HLLC, STAGE, TX>(a, rows, blockIdx.x);
}

// This thread's share of d L / d eta of both stages (eta1, eta2: their
// edge_eta), edge by edge, each stage's sum in item order.
__device__ void eta_parts(const GridDesc& d, const double* eta1, const double* eta2, int len, double* acc1, double* acc2) {
    double s1 = 0.0, s2 = 0.0;
    for (int e = 0; e < 4; ++e) {
        if (d.bc[e] != BC_TIDAL) continue;
        const int n = e < 2 ? d.ny : d.nx;
#pragma unroll 4
        for (int i = threadIdx.x; i < 2 * n; i += 1024) {
            const long long o = edge_slot(e, i >= n, i >= n ? i - n : i, len);
            s1 = s1 + eta1[o];
            s2 = s2 + eta2[o];
        }
    }
    *acc1 = s1;
    *acc2 = s2;
}

// Gauges of a session: cells (eta = h + b of the cell) or bilinear
// stations (gauge_eval.hpp) with lower-left cell (gi, gj) and weights gw
// (wx then wy).
struct GaugeSpec {
    const int* gi;
    const int* gj;
    const double* gw;   // null: cell gauges
    int ng, nx, ny;
};

__device__ __forceinline__ double spec_eta(const GaugeSpec& G, const double* h, const double* bed, long long pitch,
                                           int k) {
    if (G.gw == nullptr) {
        const long long o = (long long)G.gj[k] * pitch + G.gi[k];
        return h[o] + bed[o];
    }
    return station_eta(h, bed, pitch, G.nx, G.ny, G.gi[k], G.gj[k], G.gw[k], G.gw[G.ng + k]);
}

// Gauge misfit of one state: loss += sum_k (eta_k - target_k)^2, eta
// recorded per gauge; a single workgroup, fixed summation order.
struct LossArgs {
    const double* h;
    const double* bed;
    long long pitch;
    GaugeSpec G;
    const double* tgt;          // nsteps x ng
    double* eta;                // nsteps x ng
    double* loss;
};

__device__ __forceinline__ void gauge_loss(const LossArgs& A, int step) {
    __shared__ double red[256];
    double acc = 0.0;
    const int ng = A.G.ng;
    const double* tgt = A.tgt + (long long)step * ng;
    double* eta = A.eta + (long long)step * ng;
    for (int k = threadIdx.x; k < ng; k += 256) {
        const double e = spec_eta(A.G, A.h, A.bed, A.pitch, k);
        eta[k] = e;
        const double m = e - tgt[k];
        acc = acc + m * m;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] = red[threadIdx.x] + red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) *A.loss = *A.loss + red[0];
}

__global__ __launch_bounds__(256) void k_gauge_loss(LossArgs A, int step) { gauge_loss(A, step); }

// Seeds d L / d U^{n+1} at the gauges.  One thread per distinct gauge cell
// (cell_pos[u]) adds its taps (cell_gauges[q], weight cell_w[q] for q in
// cell_start[u] .. cell_start[u+1]) in gauge order, as a single thread
// walking all gauges would.  A cell gauge has one tap of weight 1; a
// station the four of its bilinear weights ((1-wx)(1-wy), wx(1-wy),
// (1-wx)wy, wx wy), since d eta / d h = d eta / d b = weight there.
struct SeedArgs {
    const double* h;            // U^{n+1}
    const double* bed;
    long long pitch;
    GaugeSpec G;
    const double* tgt;          // the step's targets
    const int* cell_start;
    const int* cell_gauges;
    const double* cell_w;
    const long long* cell_pos;
    int ncells;
    double scale;
    double* lam_h;
    double* grad_b;
};

__device__ __forceinline__ void gauge_seed(const SeedArgs& A, int blk) {
    const double* __restrict__ h = A.h;
    const double* __restrict__ bed = A.bed;
    const long long pitch = A.pitch;
    const GaugeSpec& G = A.G;
    const double* __restrict__ tgt = A.tgt;
    const int* __restrict__ cell_start = A.cell_start;
    const int* __restrict__ cell_gauges = A.cell_gauges;
    const double* __restrict__ cell_w = A.cell_w;
    const double scale = A.scale;
    double* __restrict__ lam_h = A.lam_h;
    double* __restrict__ grad_b = A.grad_b;
    const int u = blk * 256 + threadIdx.x;
    if (u >= A.ncells) return;
    const long long* __restrict__ cell_pos = A.cell_pos;
    const long long o = cell_pos[u];
    double lh = lam_h[o], gb = grad_b[o];
    for (int q = cell_start[u]; q < cell_start[u + 1]; ++q) {
        const int k = cell_gauges[q];
        const double e = spec_eta(G, h, bed, pitch, k);
        double sk = 2.0 * scale * (e - tgt[k]);
        if (G.gw != nullptr) sk = sk * cell_w[q];
        lh += sk;
        gb += sk;
    }
    lam_h[o] = lh;
    grad_b[o] = gb;
}

__global__ __launch_bounds__(256) void k_gauge_seed(SeedArgs A) { gauge_seed(A, blockIdx.x); }



// Scalar part of the reverse of one step (one workgroup).  scal[0] is the
// adjoint of t_{s+1} carried from later steps, scal[1] that of a dt that
// the next step reused.  Adds d L / d dt * d dt / d U at the cell of
// maximum speed to lam (the adjoint of U_s) when dt was the CFL dt.
struct DtArgs {
    GridDesc d;                 // stage 1 (input U_s)
    const double* hist;
    const double* part_dt;      // 2 x nbody partial sums of d L / d dt
    int nbody;
    const double* edge_eta;     // of stage 1, then of stage 2
    int edge_len;
    const double* pval;
    const long long* pidx;
    int nargmax;
    double* lam;                // the adjoint of U_s
    double* scal;
};

__device__ __forceinline__ void dt_rev(const DtArgs& A) {
    const GridDesc& d = A.d;
    const double* hist = A.hist;
    const double* part_dt = A.part_dt;
    const int nbody = A.nbody;
    const double* edge_eta = A.edge_eta;
    const int edge_len = A.edge_len;
    const double* pval = A.pval;
    const long long* pidx = A.pidx;
    const int nargmax = A.nargmax;
    double* lam = A.lam;
    double* scal = A.scal;
    __shared__ double red[3][1024];
    __shared__ double sv[1024];
    __shared__ long long si[1024];
    __shared__ double tide[2];   // eta'(t), eta'(t + dt)
    const double t = hist[0], dt = hist[1];
    // The kernel is bound by dependent memory round trips: each loop below
    // issues four elements' loads before it waits, and adds or compares them
    // in the element order of a plain strided loop.
    double a = 0.0;
    for (int i0 = threadIdx.x; i0 < 2 * nbody; i0 += 4 * 1024) {
        double v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = part_dt[min(i0 + u * 1024, 2 * nbody - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i0 + u * 1024 < 2 * nbody) a = a + v[u];
    }
    double best = 0.0;
    long long bi = -1;
    for (int i0 = threadIdx.x; i0 < nargmax; i0 += 4 * 1024) {
        double v[4];
        long long x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = min(i0 + u * 1024, nargmax - 1);
            v[u] = pval[i];
            x[u] = pidx[i];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i0 + u * 1024 < nargmax && (v[u] > best || (v[u] == best && x[u] >= 0 && (bi < 0 || x[u] < bi)))) {
                best = v[u];
                bi = x[u];
            }
    }
    red[0][threadIdx.x] = a;
    sv[threadIdx.x] = best;
    si[threadIdx.x] = bi;
    const int w = threadIdx.x / WAVE;
    if (w < 2) {
        const double v = adj::tidal_deta(d, w ? t + dt : t);
        if (threadIdx.x % WAVE == 0) tide[w] = v;
    }
    // d L / d eta_tidal of stage 1 (at t) and of stage 2 (at t + dt)
    eta_parts(d, edge_eta, edge_eta + edge_slot(4, 0, 0, edge_len), edge_len, &red[1][threadIdx.x], &red[2][threadIdx.x]);
    __syncthreads();
    // a tree over the workgroup: its upper levels in LDS, the last wavefront's
    // by lane shuffles
    auto later = [](double v, long long x, double& best, long long& bi) {
        if (v > best || (v == best && x >= 0 && (bi < 0 || x < bi))) {
            best = v;
            bi = x;
        }
    };
    for (int s = 512; s >= WAVE; s >>= 1) {
        if (threadIdx.x < s) {
            for (int q = 0; q < 3; ++q) red[q][threadIdx.x] = red[q][threadIdx.x] + red[q][threadIdx.x + s];
            later(sv[threadIdx.x + s], si[threadIdx.x + s], sv[threadIdx.x], si[threadIdx.x]);
        }
        __syncthreads();
    }
    if (threadIdx.x >= WAVE) return;
    double r0 = red[0][threadIdx.x], r1 = red[1][threadIdx.x], r2 = red[2][threadIdx.x];
    double ms = sv[threadIdx.x];
    long long mi = si[threadIdx.x];
    for (int s = WAVE / 2; s > 0; s >>= 1) {
        r0 = r0 + __shfl_down(r0, s, WAVE);
        r1 = r1 + __shfl_down(r1, s, WAVE);
        r2 = r2 + __shfl_down(r2, s, WAVE);
        const double v = __shfl_down(ms, s, WAVE);
        const long long x = __shfl_down(mi, s, WAVE);
        later(v, x, ms, mi);
    }
    if (threadIdx.x != 0) return;
    const bool recomputed = hist[2] != 0.0;
    const double lam_t1 = scal[0] + r2 * tide[1];   // stage 2 ran at t + dt
    const double gdt = r0 + lam_t1 + scal[1];
    double lam_t = lam_t1 + r1 * tide[0];
    double carry = 0.0;
    const double dt_max = d.t_end - t;
    if (d.dt_fixed > 0.0) {
        if (!(d.dt_fixed < dt_max)) lam_t -= gdt;           // dt = t_end - t
    } else if (recomputed) {
        double dc = ms > 0.0 ? d.cfl / ms : d.cfl * dmin(d.dx, d.dy) / sqrt(d.g * DRY_TOLERANCE);
        dc = dc * d.ssp_coeff;
        if (!(dc < dt_max)) {
            lam_t -= gdt;                                    // dt = t_end - t
        } else if (ms > 0.0 && mi >= 0) {                    // dt = cfl ssp / max speed
            const long long idx = mi;
            const long long k = (idx / d.nx) * d.pitch + idx % d.nx;
            const double l0 = lam[k], l1 = lam[d.plane + k], l2 = lam[2 * d.plane + k];
            const double lms = gdt * (-(d.cfl * d.ssp_coeff) / (ms * ms));
            const adj::S3 l = adj::cfl_speed_rev(d.g, d.dx, d.dy, d.ah[k], d.ahu[k], d.ahv[k], lms);
            lam[k] = l0 + l.h;
            lam[d.plane + k] = l1 + l.hu;
            lam[2 * d.plane + k] = l2 + l.hv;
        }
    } else {
        carry = gdt;                                         // dt reused from the step before
    }
    scal[0] = lam_t;
    scal[1] = carry;
}

__global__ __launch_bounds__(1024) void k_dt_rev(DtArgs A) { dt_rev(A); }

// ---------------------------------------------------------------------
// Batched runs and sweeps over several sessions: each kernel below is one
// launch over the blocks of every member, in the members' own block
// decomposition (a table entry names the member and its block), so that a
// member's arithmetic and sums are exactly those of its single-session
// sweep.

// A block of one member: the member, the block's index within the member's
// launch and that launch's block count.
struct BlockRef {
    int member, blk, nblk, pad;
};

// REC: recording (the replay of a sweep), else a step of the forward run.
template <int STAGE, bool HLLC, bool REC>
__global__ __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(RKG_WAVES_PER_EU, 8))) void k_step_batch(
    const GridDesc* __restrict__ descs, const BatchTile* __restrict__ tiles, const int* __restrict__ parity) {
    __shared__ TileRing ring;
    const BatchTile t = tiles[xcd_tile(blockIdx.x, gridDim.x)];
    const GridDesc& d = descs[t.member];
    stage_tile<STAGE, HLLC, true, REC, BatchTile>(d, ring, parity[t.member], MODE_STEP, d.t_end, t);
}

__global__ __launch_bounds__(256) void k_gauge_loss_batch(const LossArgs* __restrict__ la, int step) {
    gauge_loss(la[blockIdx.x], step);
}

__global__ __launch_bounds__(256) void k_gauge_seed_batch(const SeedArgs* __restrict__ sa,
                                                         const BlockRef* __restrict__ tab) {
    const BlockRef r = tab[blockIdx.x];
    gauge_seed(sa[r.member], r.blk);
}

template <int STAGE>
__global__ __launch_bounds__(256) void k_adj_body_batch(const AdjStage* __restrict__ as,
                                                       const BlockRef* __restrict__ tab) {
    const BlockRef r = tab[blockIdx.x];
    adj_body<STAGE>(as[r.member], r.blk, r.nblk);
}

// The tidal-edge variants (TY, TX) serve every member: they only add the
// bookkeeping of tidal ghost cells, which other edges do not produce.
template <bool HLLC, int STAGE>
__global__ __launch_bounds__(WAVE) void k_adj_y_batch(const AdjStage* __restrict__ as,
                                                     const BlockRef* __restrict__ tab) {
    __shared__ alignas(16) YRows rows;
    const BlockRef r = tab[xcd_tile(blockIdx.x, gridDim.x)];
    adj_y<HLLC, STAGE, true>(as[r.member], rows, r.blk);
}

template <bool HLLC, int STAGE>
__global__ __launch_bounds__(WAVE) void k_adj_x_batch(const AdjStage* __restrict__ as,
                                                     const BlockRef* __restrict__ tab) {
    __shared__ alignas(16) XRows rows;
    const BlockRef r = tab[blockIdx.x];
    adj_x<HLLC, STAGE, true>(as[r.member], rows, r.blk);
}

__global__ __launch_bounds__(1024) void k_dt_rev_batch(const DtArgs* __restrict__ da) { dt_rev(da[blockIdx.x]); }

// Still-water initial state: h = max(eta0 - b, 0) and its bed adjoint.
__global__ __launch_bounds__(256) void k_fold_still_water(const double* __restrict__ bed, const double* __restrict__ lam_h,
                                                         double eta0, int nx, int ny, long long pitch,
                                                         double* __restrict__ grad_b) {
    const long long n = (long long)nx * ny;
    for (long long idx = blockIdx.x * 256ll + threadIdx.x; idx < n; idx += (long long)gridDim.x * 256) {
        const long long k = (idx / nx) * pitch + idx % nx;
        if (eta0 - bed[k] > 0.0) grad_b[k] -= lam_h[k];
    }
}

}  // namespace

struct rkg_adjoint {
    unsigned magic;
    rkg_grid* g;
    int nsteps, K, nseg, ng;
    int* gi;                    // device
    int* gj;
    double* gw;                 // device: station weights wx then wy, or null (cell gauges)
    int* cell_start;            // device CSR of the distinct gauge cells (ncells + 1)
    int* cell_gauges;           // device: gauge of each tap, per cell in gauge order
    double* cell_w;             // device: weight of each tap (stations)
    long long* cell_pos;        // device: offset of each distinct cell in a plane
    int ncells;
    double* tgt;                // device, nsteps x ng
    double* eta;                // device, nsteps x ng (gauge eta of the last forward run)
    double* ckpt;               // nseg x 3 planes
    CtrlSlot* ckpt_ctrl;        // nseg x 2 (device)
    std::vector<int> ckpt_parity;
    double* ws;                 // segment workspace: A (K+1) x 3, B K x 3, div1 K x 3, div2 K x 3
    double* lam;                // lamA (3), lamB (3), lamDiv (3), grad_b, grad_n
    double* hist;               // K x HIST
    double* part;               // part_dt (2 x body blocks), argmax values
    long long* part_idx;        // argmax cells
    double* scal;               // adjoint of the clock and of a reused dt
    double* edge_eta;           // edge_eta of stage 1, then of stage 2 (edge_slot)
    int edge_len;
    double* loss_dev;
    double* loss_host;
    char* batch_host;           // argument tables of batched calls that this session leads (pinned
    char* batch_dev;            // and on the device), grown as needed
    size_t batch_bytes;
    CtrlSlot end_ctrl[2];
    int end_parity;
    bool have_forward;
    float fwd_ms, bwd_ms;
    hipEvent_t ev[2];
    // Overlapped replay (rkg_adjoint_backward): a second workspace and
    // history, so that segment s - 1 is replayed on rstream while segment s
    // is reversed on the grid's stream.  ws / hist and ws_alt / hist_alt
    // swap as the sweep moves between the sets; cur_set is the set in ws.
    double* ws_alt;
    double* hist_alt;
    int cur_set;
    bool overlap_off;           // the second set did not fit, or a single segment
    hipStream_t rstream;
    hipEvent_t seg_ev[4];       // replay into set 0 / 1 done, reverse of set 0 / 1 done
};

namespace {

// A live session on a live grid (the grid may have been destroyed by its
// caller while the session still holds its device state: then only
// rkg_adjoint_destroy is accepted).
bool valid(const rkg_adjoint* a) {
    if (a == nullptr || a->magic != ADJ_MAGIC) return false;
    if (!grid_valid(a->g)) {
        set_error("the grid of this adjoint session has been destroyed");
        return false;
    }
    return true;
}

size_t P(const rkg_adjoint* a) { return a->g->plane; }
double* wsA(rkg_adjoint* a, int k) { return a->ws + (size_t)k * 3 * P(a); }
double* wsB(rkg_adjoint* a, int k) { return a->ws + (size_t)(a->K + 1 + k) * 3 * P(a); }
double* wsD1(rkg_adjoint* a, int k) { return a->ws + (size_t)(2 * a->K + 1 + k) * 3 * P(a); }
double* wsD2(rkg_adjoint* a, int k) { return a->ws + (size_t)(3 * a->K + 1 + k) * 3 * P(a); }
double* lamA(rkg_adjoint* a) { return a->lam; }
double* lamB(rkg_adjoint* a) { return a->lam + 3 * P(a); }
double* lamDiv(rkg_adjoint* a) { return a->lam + 6 * P(a); }
double* gradB(rkg_adjoint* a) { return a->lam + 9 * P(a); }
double* gradN(rkg_adjoint* a) { return a->lam + 10 * P(a); }

GridDesc stage_desc(rkg_adjoint* a, double* in, double* in2, double* out2) {
    GridDesc d = make_desc(a->g);
    d.ah = in; d.ahu = in + P(a); d.ahv = in + 2 * P(a);
    d.bh = in2; d.bhu = in2 + P(a); d.bhv = in2 + 2 * P(a);
    d.o2h = out2; d.o2hu = out2 + P(a); d.o2hv = out2 + 2 * P(a);
    d.sh = d.shu = d.shv = nullptr;
    d.mpart = nullptr;
    return d;
}

template <int STAGE>
void launch_rec(rkg_grid* g, const GridDesc& d, int p, hipStream_t st) {
    const int ntiles = d.ntiles;
    const double tlim = g->cfg.t_end;
    if (g->cfg.use_hllc)
        hipLaunchKernelGGL((k_stage<STAGE, true, true, true>), dim3(ntiles), dim3(WAVE), 0, st, d, p, MODE_STEP, tlim);
    else
        hipLaunchKernelGGL((k_stage<STAGE, false, true, true>), dim3(ntiles), dim3(WAVE), 0, st, d, p, MODE_STEP, tlim);
}

// Workgroups of k_adj_x, and how many of them, the first, hold an edge strip.
int x_blocks(int nx, int ny) { return ((nx + AW - 1) / AW) * ((ny + XROWS - 1) / XROWS); }
int x_edge_blocks(int nx, int ny) { return std::min(x_blocks(nx, ny), 2 * ((ny + XROWS - 1) / XROWS)); }

// The stage's face reverse: k_adj_y then k_adj_x (both add into lam_in and
// grad_b).
template <bool HLLC, int STAGE>
void launch_faces(rkg_grid* g, const AdjStage& st) {
    const int* bc = g->cfg.bc;
    const bool tx = bc[0] == BC_TIDAL || bc[1] == BC_TIDAL, ty = bc[2] == BC_TIDAL || bc[3] == BC_TIDAL;
    const int nx = g->cfg.nx, ny = g->cfg.ny;
    const int yblocks = ((nx + WAVE - 1) / WAVE) * ((ny + st.ty - 1) / st.ty);
    const int xblocks = x_blocks(nx, ny);
    if (ty)
        hipLaunchKernelGGL((k_adj_y<HLLC, STAGE, true>), dim3(yblocks), dim3(WAVE), 0, g->stream, st);
    else
        hipLaunchKernelGGL((k_adj_y<HLLC, STAGE, false>), dim3(yblocks), dim3(WAVE), 0, g->stream, st);
    if (tx)
        hipLaunchKernelGGL((k_adj_x<HLLC, STAGE, true>), dim3(xblocks), dim3(WAVE), 0, g->stream, st);
    else
        hipLaunchKernelGGL((k_adj_x<HLLC, STAGE, false>), dim3(xblocks), dim3(WAVE), 0, g->stream, st);
}

int body_blocks(const rkg_grid* g) {
    const long long n = (long long)g->cfg.nx * g->cfg.ny;
    return (int)std::min<long long>((n + 255) / 256, 2048);
}


}  // namespace

namespace {

// A session over gauges given as lower-left cells gauge_i / gauge_j and, for
// stations, the weights wx / wy (null for cell gauges).
int create_session(rkg_grid* g, int nsteps, int K, int ng, const int* gauge_i, const int* gauge_j,
                   const double* wx, const double* wy, const double* targets, rkg_adjoint** out) {
    if (g->scheme != RKG_TIME_RK2) {
        set_error("the adjoint is that of the SSP-RK2 step; set time scheme rk2");
        return RKG_ERR_UNSUPPORTED;
    }
    if (g->forcing) {
        set_error("the adjoint does not cover the surface forcing; switch it off");
        return RKG_ERR_UNSUPPORTED;
    }
    if (sponge_on(g)) {
        set_error("the adjoint does not cover the sponge relaxation; set its width to 0");
        return RKG_ERR_UNSUPPORTED;
    }
    for (int e = 0; e < 4; ++e)
        if (g->cfg.bc[e] == RKG_BC_CHAPMAN) {
            set_error("the adjoint does not cover Chapman edges");
            return RKG_ERR_UNSUPPORTED;
        }
    int rc = rkg_use_manning_field(g, 1);
    if (rc) return rc;
    rkg_adjoint* a = new rkg_adjoint();
    memset((void*)a, 0, sizeof *a);
    a->ckpt_parity = std::vector<int>();
    a->g = g;
    grid_retain(g);   // released by rkg_adjoint_destroy
    a->nsteps = nsteps;
    a->K = std::min(K, nsteps);
    a->nseg = (nsteps + a->K - 1) / a->K;
    a->ng = ng;
    a->ckpt_parity.assign(a->nseg, 0);
    const size_t Pl = g->plane;
    hipError_t e = hipSuccess;
    if (ng > 0) {
        e = hipMalloc((void**)&a->gi, ng * sizeof(int));
        if (e == hipSuccess) e = hipMalloc((void**)&a->gj, ng * sizeof(int));
        if (e == hipSuccess) e = hipMemcpy(a->gi, gauge_i, ng * sizeof(int), hipMemcpyHostToDevice);
        // taps: one per cell gauge (weight 1), four per station (its
        // bilinear weights, gauges_write :519-537); distinct cells in order
        // of first appearance, each with its taps in gauge order
        const int nx = g->cfg.nx, ny = g->cfg.ny;
        std::vector<long long> keys;
        std::vector<std::vector<std::pair<int, double>>> members;
        auto tap = [&](int k, int c, int j, double w) {
            const long long key = (long long)j * g->pitch + c;
            size_t u = 0;
            while (u < keys.size() && keys[u] != key) ++u;
            if (u == keys.size()) { keys.push_back(key); members.emplace_back(); }
            members[u].push_back({k, w});
        };
        for (int k = 0; k < ng; ++k) {
            if (!wx) { tap(k, gauge_i[k], gauge_j[k], 1.0); continue; }
            const int c0 = gauge_i[k], j0 = gauge_j[k];
            const int c1 = std::min(c0 + 1, nx - 1), j1 = std::min(j0 + 1, ny - 1);
            tap(k, c0, j0, (1.0 - wx[k]) * (1.0 - wy[k]));
            tap(k, c1, j0, wx[k] * (1.0 - wy[k]));
            tap(k, c0, j1, (1.0 - wx[k]) * wy[k]);
            tap(k, c1, j1, wx[k] * wy[k]);
        }
        std::vector<int> start(1, 0), list;
        std::vector<double> wlist;
        for (const auto& m : members) {
            for (const auto& t : m) { list.push_back(t.first); wlist.push_back(t.second); }
            start.push_back((int)list.size());
        }
        a->ncells = (int)keys.size();
        if (e == hipSuccess) e = hipMalloc((void**)&a->cell_start, start.size() * sizeof(int));
        if (e == hipSuccess) e = hipMalloc((void**)&a->cell_gauges, list.size() * sizeof(int));
        if (e == hipSuccess) e = hipMalloc((void**)&a->cell_w, wlist.size() * sizeof(double));
        if (e == hipSuccess) e = hipMalloc((void**)&a->cell_pos, keys.size() * sizeof(long long));
        if (e == hipSuccess) e = hipMemcpy(a->cell_start, start.data(), start.size() * sizeof(int), hipMemcpyHostToDevice);
        if (e == hipSuccess) e = hipMemcpy(a->cell_gauges, list.data(), list.size() * sizeof(int), hipMemcpyHostToDevice);
        if (e == hipSuccess) e = hipMemcpy(a->cell_w, wlist.data(), wlist.size() * sizeof(double), hipMemcpyHostToDevice);
        if (e == hipSuccess) e = hipMemcpy(a->cell_pos, keys.data(), keys.size() * sizeof(long long), hipMemcpyHostToDevice);
        if (wx) {
            std::vector<double> w(wx, wx + ng);
            w.insert(w.end(), wy, wy + ng);
            if (e == hipSuccess) e = hipMalloc((void**)&a->gw, 2 * (size_t)ng * sizeof(double));
            if (e == hipSuccess) e = hipMemcpy(a->gw, w.data(), 2 * (size_t)ng * sizeof(double), hipMemcpyHostToDevice);
        }
        if (e == hipSuccess) e = hipMemcpy(a->gj, gauge_j, ng * sizeof(int), hipMemcpyHostToDevice);
        if (e == hipSuccess) e = hipMalloc((void**)&a->tgt, (size_t)nsteps * ng * sizeof(double));
        if (e == hipSuccess) e = hipMalloc((void**)&a->eta, (size_t)nsteps * ng * sizeof(double));
        if (e == hipSuccess) e = hipMemset(a->tgt, 0, (size_t)nsteps * ng * sizeof(double));
        if (e == hipSuccess && targets)
            e = hipMemcpy(a->tgt, targets, (size_t)nsteps * ng * sizeof(double), hipMemcpyHostToDevice);
    }
    if (e == hipSuccess) e = hipMalloc((void**)&a->ckpt, (size_t)a->nseg * 3 * Pl * sizeof(double));
    if (e == hipSuccess) e = hipMalloc((void**)&a->ckpt_ctrl, (size_t)a->nseg * 2 * sizeof(CtrlSlot));
    if (e == hipSuccess) e = hipMalloc((void**)&a->ws, (size_t)(12 * a->K + 3) * Pl * sizeof(double));
    if (e == hipSuccess) e = hipMalloc((void**)&a->lam, 11 * Pl * sizeof(double));
    if (e == hipSuccess) e = hipMalloc((void**)&a->hist, (size_t)a->K * HIST * sizeof(double));
    a->edge_len = std::max(g->cfg.nx, g->cfg.ny);
    if (e == hipSuccess)
        e = hipMalloc((void**)&a->part, (size_t)(3 * body_blocks(g)) * sizeof(double));   // part_dt, argmax values
    if (e == hipSuccess) e = hipMalloc((void**)&a->edge_eta, 2 * (size_t)edge_slot(4, 0, 0, a->edge_len) * sizeof(double));
    if (e == hipSuccess) e = hipMemset(a->edge_eta, 0, 2 * (size_t)edge_slot(4, 0, 0, a->edge_len) * sizeof(double));
    if (e == hipSuccess) e = hipMalloc((void**)&a->part_idx, (size_t)body_blocks(g) * sizeof(long long));
    if (e == hipSuccess) e = hipMalloc((void**)&a->scal, 2 * sizeof(double));
    if (e == hipSuccess) e = hipMalloc((void**)&a->loss_dev, sizeof(double));
    if (e == hipSuccess) e = hipHostMalloc((void**)&a->loss_host, sizeof(double), hipHostMallocDefault);
    if (e == hipSuccess) e = hipMemset(a->ws, 0, (size_t)(12 * a->K + 3) * Pl * sizeof(double));
    if (e == hipSuccess) e = hipMemset(a->lam, 0, 11 * Pl * sizeof(double));
    if (e == hipSuccess) e = hipEventCreate(&a->ev[0]);
    if (e == hipSuccess) e = hipEventCreate(&a->ev[1]);
    a->magic = ADJ_MAGIC;
    if (e != hipSuccess) {
        set_error("adjoint allocation failed: %s", hipGetErrorString(e));
        rkg_adjoint_destroy(&a);
        return RKG_ERR_HIP;
    }
    *out = a;
    return RKG_OK;
}

}  // namespace

extern "C" {

int rkg_adjoint_create(rkg_grid* g, int nsteps, int K, int ng, const int* gauge_i, const int* gauge_j,
                       const double* targets, rkg_adjoint** out) {
    if (!out) { set_error("null argument"); return RKG_ERR_RANGE; }
    *out = nullptr;
    if (!grid_valid(g)) return RKG_ERR_BAD_HANDLE;
    if (nsteps < 1 || K < 1 || ng < 0 || (ng > 0 && (!gauge_i || !gauge_j))) {
        set_error("need nsteps >= 1, checkpoint_interval >= 1 and gauge indices");
        return RKG_ERR_RANGE;
    }
    for (int k = 0; k < ng; ++k)
        if (gauge_i[k] < 0 || gauge_i[k] >= g->cfg.nx || gauge_j[k] < 0 || gauge_j[k] >= g->cfg.ny) {
            set_error("gauge %d at (%d, %d) lies outside the %dx%d grid", k, gauge_i[k], gauge_j[k], g->cfg.nx,
                      g->cfg.ny);
            return RKG_ERR_RANGE;
        }
    return create_session(g, nsteps, K, ng, gauge_i, gauge_j, nullptr, nullptr, targets, out);
}

int rkg_adjoint_create_stations(rkg_grid* g, int nsteps, int K, int n, const double* x, const double* y,
                                const double* targets, rkg_adjoint** out) {
    if (!out) { set_error("null argument"); return RKG_ERR_RANGE; }
    *out = nullptr;
    if (!grid_valid(g)) return RKG_ERR_BAD_HANDLE;
    if (nsteps < 1 || K < 1 || n < 0 || n > RKG_MAX_GAUGES || (n > 0 && (!x || !y))) {
        set_error("need nsteps >= 1, checkpoint_interval >= 1 and station coordinates");
        return RKG_ERR_RANGE;
    }
    std::vector<int> ci(n), cj(n);
    std::vector<double> wx(n), wy(n);
    for (int k = 0; k < n; ++k)
        if (!station_weights(g->cfg, x[k], y[k], &ci[k], &cj[k], &wx[k], &wy[k])) {
            set_error("station %d at (%g, %g) m lies outside the domain", k, x[k], y[k]);
            return RKG_ERR_RANGE;
        }
    return create_session(g, nsteps, K, n, ci.data(), cj.data(), wx.data(), wy.data(), targets, out);
}

void rkg_adjoint_destroy(rkg_adjoint** pa) {
    if (!pa || !*pa) return;
    rkg_adjoint* a = *pa;
    if (a->magic != ADJ_MAGIC) { *pa = nullptr; return; }
    if (a->g && a->g->stream) (void)hipStreamSynchronize(a->g->stream);
    if (a->rstream) (void)hipStreamSynchronize(a->rstream);
    for (void* p : {(void*)a->gi, (void*)a->gj, (void*)a->gw, (void*)a->cell_start, (void*)a->cell_gauges,
                    (void*)a->cell_w, (void*)a->cell_pos, (void*)a->tgt, (void*)a->eta, (void*)a->ckpt, (void*)a->ckpt_ctrl,
                    (void*)a->ws, (void*)a->lam, (void*)a->hist, (void*)a->loss_dev, (void*)a->part,
                    (void*)a->part_idx, (void*)a->scal, (void*)a->edge_eta, (void*)a->ws_alt, (void*)a->hist_alt})
        if (p) (void)hipFree(p);
    if (a->rstream) (void)hipStreamDestroy(a->rstream);
    for (hipEvent_t ev : a->seg_ev)
        if (ev) (void)hipEventDestroy(ev);
    if (a->loss_host) (void)hipHostFree(a->loss_host);
    if (a->batch_host) (void)hipHostFree(a->batch_host);
    if (a->batch_dev) (void)hipFree(a->batch_dev);
    if (a->ev[0]) (void)hipEventDestroy(a->ev[0]);
    if (a->ev[1]) (void)hipEventDestroy(a->ev[1]);
    rkg_grid* g = a->g;
    a->magic = ADJ_DEAD;
    delete a;
    *pa = nullptr;
    if (g) grid_release(g);
}

int rkg_adjoint_set_targets(rkg_adjoint* a, const double* targets) {
    if (!valid(a)) return RKG_ERR_BAD_HANDLE;
    if (a->ng == 0) return RKG_OK;
    if (!targets) return RKG_ERR_RANGE;
    HIP_TRY(hipMemcpy(a->tgt, targets, (size_t)a->nsteps * a->ng * sizeof(double), hipMemcpyHostToDevice));
    return RKG_OK;
}

int rkg_adjoint_gauge_eta(rkg_adjoint* a, double* eta) {
    if (!valid(a)) return RKG_ERR_BAD_HANDLE;
    if (!a->have_forward) { set_error("no forward run yet"); return RKG_ERR_NOT_READY; }
    if (a->ng == 0) return RKG_OK;
    if (!eta) return RKG_ERR_RANGE;
    HIP_TRY(hipMemcpy(eta, a->eta, (size_t)a->nsteps * a->ng * sizeof(double), hipMemcpyDeviceToHost));
    return RKG_OK;
}

}  // extern "C"

namespace {

GaugeSpec gauge_spec(const rkg_adjoint* a) {
    return GaugeSpec{a->gi, a->gj, a->gw, a->ng, a->g->cfg.nx, a->g->cfg.ny};
}

// --- the forward run and the reverse sweep, as per-step pieces that queue
// work on the session's stream without waiting, so that several sessions on
// several streams can be interleaved step by step ---------------------------

int fwd_begin(rkg_adjoint* a) {
    rkg_grid* g = a->g;
    if (g->scheme != RKG_TIME_RK2) {
        set_error("the adjoint is that of the SSP-RK2 step; set time scheme rk2");
        return RKG_ERR_UNSUPPORTED;
    }
    if (g->forcing) {
        set_error("the adjoint does not cover the surface forcing; switch it off");
        return RKG_ERR_UNSUPPORTED;
    }
    if (sponge_on(g)) {
        set_error("the adjoint does not cover the sponge relaxation; set its width to 0");
        return RKG_ERR_UNSUPPORTED;
    }
    for (int e = 0; e < 4; ++e)
        if (g->cfg.bc[e] == RKG_BC_CHAPMAN) {
            set_error("the adjoint does not cover Chapman edges");
            return RKG_ERR_UNSUPPORTED;
        }
    HIP_TRY(hipMemsetAsync(a->loss_dev, 0, sizeof(double), g->stream));
    HIP_TRY(hipEventRecord(a->ev[0], g->stream));
    return RKG_OK;
}

LossArgs loss_args(rkg_adjoint* a) {
    rkg_grid* g = a->g;
    return LossArgs{g->buf, g->buf + 6 * g->plane, (long long)g->pitch, gauge_spec(a), a->tgt, a->eta, a->loss_dev};
}

// The checkpoint of segment s, the state before step s K, on stream st.
int fwd_checkpoint(rkg_adjoint* a, int s, hipStream_t st) {
    rkg_grid* g = a->g;
    const size_t Pl = g->plane;
    HIP_TRY(hipMemcpyAsync(a->ckpt + (size_t)s * 3 * Pl, g->buf, 3 * Pl * sizeof(double), hipMemcpyDeviceToDevice, st));
    HIP_TRY(hipMemcpyAsync(a->ckpt_ctrl + 2 * s, g->ctrl, 2 * sizeof(CtrlSlot), hipMemcpyDeviceToDevice, st));
    a->ckpt_parity[s] = g->parity;
    return RKG_OK;
}

// Step n of the forward run: the checkpoint at a segment start, the step,
// the gauge misfit.
int fwd_step(rkg_adjoint* a, int n) {
    rkg_grid* g = a->g;
    int rc = RKG_OK;
    if (n % a->K == 0) {
        if (g->speed_stale) rc = rkg_step(g, 0);   // make the control slot current before saving it
        if (!rc) rc = fwd_checkpoint(a, n / a->K, g->stream);
        if (rc) return rc;
    }
    rc = rkg_step(g, 1);
    if (rc) return rc;
    if (a->ng > 0)
        hipLaunchKernelGGL(k_gauge_loss, dim3(1), dim3(256), 0, g->stream, loss_args(a), n);
    return RKG_OK;
}

int fwd_end(rkg_adjoint* a) {
    rkg_grid* g = a->g;
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipEventRecord(a->ev[1], g->stream));
    HIP_TRY(hipMemcpyAsync(a->end_ctrl, g->ctrl, 2 * sizeof(CtrlSlot), hipMemcpyDeviceToHost, g->stream));
    HIP_TRY(hipMemcpyAsync(a->loss_host, a->loss_dev, sizeof(double), hipMemcpyDeviceToHost, g->stream));
    return RKG_OK;
}

// After the stream has drained.
int fwd_finish(rkg_adjoint* a, double* loss) {
    HIP_TRY(hipEventElapsedTime(&a->fwd_ms, a->ev[0], a->ev[1]));
    a->end_parity = a->g->parity;
    a->have_forward = true;
    if (loss) *loss = *a->loss_host;
    return RKG_OK;
}

// Per-sweep settings of one session.
struct BwdPlan {
    int tile_rows, nb, nargmax;
    bool cfl_dt;
    long long edge_size;
    double scale;
    int p;                      // parity of the replay
};

// Rows per workgroup of k_adj_y for a launch over `rows` rows of 64 columns:
// about 2048 workgroups, two waves on each of the 1024 SIMDs (1024^2 basin,
// us: 8 rows 48, 7 rows 57, 10 rows 56).  The remainder tiles of the strips may
// make it a few more; a row more per tile, to stay within 2048, is slower
// (897x1773, 13 rows and 2055 workgroups 70, 14 rows 73; 1947x1453, 22 rows and
// 2077 workgroups 112, 23 rows 114).
int adj_y_rows(long long rows) { return (int)std::min<long long>(32, std::max<long long>(4, (rows + 2047) / 2048)); }

int bwd_begin(rkg_adjoint* a, double loss_scale, int tile_rows, BwdPlan& pl) {
    if (!a->have_forward) { set_error("rkg_adjoint_backward before rkg_adjoint_forward"); return RKG_ERR_NOT_READY; }
    rkg_grid* g = a->g;
    const long long ny = g->cfg.ny;
    const long long ystrips = (g->cfg.nx + WAVE - 1) / WAVE;
    if (tile_rows <= 0) tile_rows = adj_y_rows(ny * ystrips);
    if (tile_rows < 4 || tile_rows > 256) { set_error("tile_rows must lie in [4, 256]"); return RKG_ERR_RANGE; }
    pl.tile_rows = tile_rows;
    pl.nb = body_blocks(g);
    pl.cfl_dt = g->cfg.dt_fixed <= 0.0;
    pl.nargmax = pl.cfl_dt ? pl.nb : 0;   // argmax partials, one per body workgroup of stage 1
    pl.edge_size = edge_slot(4, 0, 0, a->edge_len);
    pl.scale = loss_scale;
    pl.p = 0;
    const size_t Pl = g->plane;
    HIP_TRY(hipEventRecord(a->ev[0], g->stream));
    HIP_TRY(hipMemsetAsync(a->lam, 0, 11 * Pl * sizeof(double), g->stream));
    HIP_TRY(hipMemsetAsync(a->scal, 0, 2 * sizeof(double), g->stream));
    return RKG_OK;
}

int seg_steps(const rkg_adjoint* a, int s) { return std::min(a->nsteps, (s + 1) * a->K) - s * a->K; }

// Start of the replay of segment s on stream st: its checkpoint into A_0
// and the clock.
int bwd_replay_begin(rkg_adjoint* a, int s, BwdPlan& pl, hipStream_t st) {
    rkg_grid* g = a->g;
    const size_t Pl = g->plane;
    HIP_TRY(hipMemcpyAsync(wsA(a, 0), a->ckpt + (size_t)s * 3 * Pl, 3 * Pl * sizeof(double), hipMemcpyDeviceToDevice,
                           st));
    HIP_TRY(hipMemcpyAsync(g->ctrl, a->ckpt_ctrl + 2 * s, 2 * sizeof(CtrlSlot), hipMemcpyDeviceToDevice, st));
    pl.p = a->ckpt_parity[s];
    return RKG_OK;
}

// Step k of the segment's replay, recording U^n, U*, both divergences and
// the clock.
void bwd_replay_step(rkg_adjoint* a, int k, BwdPlan& pl, hipStream_t st) {
    rkg_grid* g = a->g;
    GridDesc d1 = stage_desc(a, wsA(a, k), wsB(a, k), wsA(a, k + 1));
    d1.rec = wsD1(a, k);
    d1.hist = a->hist + HIST * k;
    launch_rec<1>(g, d1, pl.p, st);
    GridDesc d2 = d1;
    d2.rec = wsD2(a, k);
    d2.hist = nullptr;
    launch_rec<2>(g, d2, pl.p, st);
    pl.p ^= 1;
}

// Puts workspace set `set` (0 or 1) in ws / hist.
void use_set(rkg_adjoint* a, int set) {
    if (set == a->cur_set) return;
    std::swap(a->ws, a->ws_alt);
    std::swap(a->hist, a->hist_alt);
    a->cur_set = set;
}

size_t ws_bytes(const rkg_adjoint* a) { return (size_t)(12 * a->K + 3) * a->g->plane * sizeof(double); }

// The second workspace, stream and events of the overlapped replay,
// allocated at the first backward sweep that can use them: a session of
// two or more segments whose second workspace takes at most half of the
// device's free memory.  Otherwise, or when an allocation fails (what was
// allocated is released), the sweeps replay on the grid's stream.
void ensure_overlap(rkg_adjoint* a) {
    if (a->rstream || a->overlap_off) return;
    a->overlap_off = true;
    if (a->nseg < 2) return;
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) { (void)hipGetLastError(); return; }
    const size_t hist_b = (size_t)a->K * HIST * sizeof(double);
    if (ws_bytes(a) + hist_b > free_b / 2) return;
    hipError_t e = hipMalloc((void**)&a->ws_alt, ws_bytes(a));
    if (e == hipSuccess) e = hipMalloc((void**)&a->hist_alt, hist_b);
    if (e == hipSuccess) e = hipMemset(a->ws_alt, 0, ws_bytes(a));
    for (int q = 0; q < 4 && e == hipSuccess; ++q) e = hipEventCreateWithFlags(&a->seg_ev[q], hipEventDisableTiming);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&a->rstream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        if (a->ws_alt) (void)hipFree(a->ws_alt);
        if (a->hist_alt) (void)hipFree(a->hist_alt);
        for (hipEvent_t& ev : a->seg_ev)
            if (ev) { (void)hipEventDestroy(ev); ev = nullptr; }
        a->ws_alt = a->hist_alt = nullptr;
        a->rstream = nullptr;
        return;
    }
    a->overlap_off = false;
}

// Arguments of the kernels that reverse step k of the current segment
// (global step n): the gauge seed, the two stages (STAGE 2 first), and the
// dt/clock kernel.
SeedArgs seed_args(rkg_adjoint* a, int k, int n, const BwdPlan& pl) {
    rkg_grid* g = a->g;
    SeedArgs A;
    A.h = wsA(a, k + 1);
    A.bed = g->buf + 6 * g->plane;
    A.pitch = (long long)g->pitch;
    A.G = gauge_spec(a);
    A.tgt = a->tgt + (size_t)n * a->ng;
    A.cell_start = a->cell_start;
    A.cell_gauges = a->cell_gauges;
    A.cell_w = a->cell_w;
    A.cell_pos = a->cell_pos;
    A.ncells = a->ncells;
    A.scale = pl.scale;
    A.lam_h = lamA(a);
    A.grad_b = gradB(a);
    return A;
}

AdjStage stage_args(rkg_adjoint* a, int k, int stage, const BwdPlan& pl) {
    const int nb = pl.nb;
    AdjStage st;
    st.lam_div = lamDiv(a);
    st.grad_b = gradB(a);
    st.grad_n = gradN(a);
    st.hist = a->hist + HIST * k;
    st.edge_len = a->edge_len;
    st.ty = pl.tile_rows;
    if (stage == 2) {   // input U* (B_k), U^n = A_k
        st.d = stage_desc(a, wsB(a, k), wsB(a, k), wsA(a, k + 1));
        st.un = wsA(a, k);
        st.div = wsD2(a, k);
        st.lam_in = lamB(a);
        st.lam_out = lamA(a);
        st.part_dt = a->part + nb;
        st.pval = nullptr;
        st.pidx = nullptr;
        st.edge_eta = a->edge_eta + pl.edge_size;
    } else {            // input U^n (A_k)
        st.d = stage_desc(a, wsA(a, k), wsB(a, k), wsA(a, k + 1));
        st.un = nullptr;
        st.div = wsD1(a, k);
        st.lam_in = lamA(a);
        st.lam_out = lamB(a);
        st.part_dt = a->part;
        st.pval = pl.cfl_dt ? a->part + 2 * nb : nullptr;
        st.pidx = pl.cfl_dt ? a->part_idx : nullptr;
        st.edge_eta = a->edge_eta;
    }
    return st;
}

DtArgs dt_args(rkg_adjoint* a, int k, const AdjStage& st1, const BwdPlan& pl) {
    DtArgs A;
    A.d = st1.d;
    A.hist = st1.hist;
    A.part_dt = a->part;
    A.nbody = pl.nb;
    A.edge_eta = a->edge_eta;
    A.edge_len = a->edge_len;
    A.pval = a->part + 2 * pl.nb;
    A.pidx = a->part_idx;
    A.nargmax = pl.nargmax;
    A.lam = lamA(a);
    A.scal = a->scal;
    return A;
}

// Reverse of step k of segment s (global step n0 + k).
void bwd_reverse_step(rkg_adjoint* a, int s, int k, const BwdPlan& pl) {
    rkg_grid* g = a->g;
    const int n = s * a->K + k;
    const int nb = pl.nb;
    if (a->ng > 0)
        hipLaunchKernelGGL(k_gauge_seed, dim3((a->ncells + 255) / 256), dim3(256), 0, g->stream,
                           seed_args(a, k, n, pl));
    const AdjStage st2 = stage_args(a, k, 2, pl);
    hipLaunchKernelGGL(k_adj_body<2>, dim3(nb), dim3(256), 0, g->stream, st2);
    if (g->cfg.use_hllc) launch_faces<true, 2>(g, st2);
    else launch_faces<false, 2>(g, st2);
    const AdjStage st1 = stage_args(a, k, 1, pl);
    hipLaunchKernelGGL(k_adj_body<1>, dim3(nb), dim3(256), 0, g->stream, st1);
    if (g->cfg.use_hllc) launch_faces<true, 1>(g, st1);
    else launch_faces<false, 1>(g, st1);
    // the step's dt and clock
    hipLaunchKernelGGL(k_dt_rev, dim3(1), dim3(1024), 0, g->stream, dt_args(a, k, st1, pl));
}

// The sweep with the replay of segment s - 1 (into workspace set (s-1)&1,
// on rstream) overlapping the reverse of segment s (set s&1, on the grid's
// stream).  Events order each set's replay before its reverse and a set's
// next replay after the reverse that last read it; the kernels and their
// inputs are those of the serial sweep, so the gradients are the same bits.
int bwd_overlapped(rkg_adjoint* a, BwdPlan& pl) {
    hipStream_t main = a->g->stream, rs = a->rstream;
    // the replays start after the work already queued on the grid's stream
    HIP_TRY(hipEventRecord(a->seg_ev[2], main));
    HIP_TRY(hipStreamWaitEvent(rs, a->seg_ev[2], 0));
    auto replay = [&](int s) -> int {
        use_set(a, s & 1);
        int rc = bwd_replay_begin(a, s, pl, rs);
        if (rc) return rc;
        for (int k = 0; k < seg_steps(a, s); ++k) bwd_replay_step(a, k, pl, rs);
        HIP_TRY(hipEventRecord(a->seg_ev[s & 1], rs));
        return RKG_OK;
    };
    int rc = replay(a->nseg - 1);
    for (int s = a->nseg - 1; s >= 0 && !rc; --s) {
        if (s > 0) {
            // set (s-1)&1 was last read by the reverse of segment s + 1
            if (s + 1 < a->nseg) HIP_TRY(hipStreamWaitEvent(rs, a->seg_ev[2 + ((s + 1) & 1)], 0));
            rc = replay(s - 1);
            if (rc) break;
        }
        HIP_TRY(hipStreamWaitEvent(main, a->seg_ev[s & 1], 0));
        use_set(a, s & 1);
        for (int k = seg_steps(a, s) - 1; k >= 0; --k) bwd_reverse_step(a, s, k, pl);
        HIP_TRY(hipEventRecord(a->seg_ev[2 + (s & 1)], main));
    }
    use_set(a, 0);
    return rc;
}

int bwd_end(rkg_adjoint* a) {
    rkg_grid* g = a->g;
    HIP_TRY(hipGetLastError());
    // the grid's control slots back to the end of the forward run
    HIP_TRY(hipMemcpyAsync(g->ctrl, a->end_ctrl, 2 * sizeof(CtrlSlot), hipMemcpyHostToDevice, g->stream));
    g->parity = a->end_parity;
    HIP_TRY(hipEventRecord(a->ev[1], g->stream));
    return RKG_OK;
}

int bwd_finish(rkg_adjoint* a) {
    HIP_TRY(hipEventElapsedTime(&a->bwd_ms, a->ev[0], a->ev[1]));
    return RKG_OK;
}

size_t al256(size_t x) { return (x + 255) / 256 * 256; }

// Bytes of argument tables that a session keeps between batched calls.  A
// sweep's grow with members times steps, 5 KB each: eight members and 20 steps take
// 0.8 MB.  Allocating 16 MB anew (16 members, 200 steps) takes 1 ms of a sweep of 57.
constexpr size_t BATCH_KEEP = (size_t)4 << 20;

void drop_tables(rkg_adjoint* a) {
    if (a->batch_host) (void)hipHostFree(a->batch_host);
    if (a->batch_dev) (void)hipFree(a->batch_dev);
    a->batch_host = a->batch_dev = nullptr;
    a->batch_bytes = 0;
}

// After a batched call, whose streams are drained.
void trim_tables(rkg_adjoint* a) {
    if (a->batch_bytes > BATCH_KEEP) drop_tables(a);
}

// Room for `bytes` of argument tables with the batch's first session.  Every
// batched call ends with its streams drained, so the last call's are free.
int batch_tables(rkg_adjoint* a, size_t bytes) {
    if (a->batch_bytes >= bytes) return RKG_OK;
    drop_tables(a);
    hipError_t e = hipHostMalloc((void**)&a->batch_host, bytes, hipHostMallocDefault);
    if (e == hipSuccess) e = hipMalloc((void**)&a->batch_dev, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        if (a->batch_host) (void)hipHostFree(a->batch_host);
        a->batch_host = nullptr;
        a->batch_dev = nullptr;
        set_error("batched adjoint: cannot allocate its %zu-byte argument tables: %s", bytes, hipGetErrorString(e));
        return RKG_ERR_HIP;
    }
    a->batch_bytes = bytes;
    return RKG_OK;
}

// Rows per stage tile by the tiles of all members: a launch serves them
// together (eight grids of 128..512 cells, us: replay stages 66 / 70 with
// each grid's own rows, 44 / 47 with these).  A height set by the caller stays.
void set_batch_tiles(int n, rkg_adjoint* const* as, GridDesc* d) {
    const int rows = rows_for([=](int r) {
        long long t = 0;
        for (int m = 0; m < n; ++m) t += grid_tiles(as[m]->g->cfg.nx, as[m]->g->cfg.ny, r);
        return t;
    }, 1);
    std::vector<int> ty(n);
    for (int m = 0; m < n; ++m) ty[m] = as[m]->g->ty == 0 ? rows : d[m].ty;
    set_launch_tiles(d, n, ty.data());
}

// The work of every stream before what the first stream queues next (to_first),
// or the work of the first before what the others queue.
hipError_t join_streams(int n, rkg_adjoint* const* as, hipEvent_t ev, bool to_first) {
    hipStream_t S = as[0]->g->stream;
    hipError_t e = hipSuccess;
    if (!to_first) e = hipEventRecord(ev, S);
    for (int m = 1; m < n && e == hipSuccess; ++m) {
        if (to_first) {
            e = hipEventRecord(ev, as[m]->g->stream);
            if (e == hipSuccess) e = hipStreamWaitEvent(S, ev, 0);
        } else {
            e = hipStreamWaitEvent(as[m]->g->stream, ev, 0);
        }
    }
    return e;
}

// Whether the forward runs of n sessions go as one: one device, one solver,
// and steps that launch the two stage kernels and nothing else; and launches
// that gain by it.  The host issues a member's step in about 16 us.  Runs of up
// to three members, and of up to six whose common launches would be of half a
// round to a round and a half of tiles, keep the chip busier on streams of their
// own, where one member's stage fills the others' tails.  us a step, streams of
// their own / as one:
//   2 x 700x600   90 / 125,  3 x 512^2    89 / 126,  3 x 1024^2  215 / 279,
//   4 x 512^2    142 / 162,  6 x 700x600 233 / 270;
//   4 x 128^2     76 /  62,  4 x 1024^2  361 / 337,  8 x 512^2   262 / 262,
//   16 x 400x300 389 / 313,  32 x 256^2  686 / 501
bool fwd_batchable(int n, rkg_adjoint* const* as) {
    long long tiles = 0;   // of 10 rows
    for (int m = 0; m < n; ++m) tiles += grid_tiles(as[m]->g->cfg.nx, as[m]->g->cfg.ny, 10);
    if (n <= 3 || (n <= 6 && tiles >= 1536 && tiles <= 3 * 1536)) return false;
    for (int m = 0; m < n; ++m) {
        const rkg_grid* g = as[m]->g;
        if (g->device != as[0]->g->device || (g->cfg.use_hllc != 0) != (as[0]->g->cfg.use_hllc != 0)) return false;
        if (!g->nfield || g->mpart || g->gauges || g->prof) return false;
    }
    return true;
}

// The forward runs of n sessions on the first session's stream: three
// launches a step (both stages and the gauge misfits of every member)
// instead of three per member, which the host could not issue as fast as the
// GPU ran them.  Every member's arithmetic is that of its own run.  `ran` is false,
// and nothing has been queued, where there is no memory for the tables.
int fwd_batched(int n, rkg_adjoint* const* as, bool& ran) {
    const bool hllc = as[0]->g->cfg.use_hllc != 0;
    const int nsteps = as[0]->nsteps, K = as[0]->K;
    hipStream_t S = as[0]->g->stream;
    std::vector<GridDesc> d(n);
    std::vector<BatchTile> tiles;
    std::vector<LossArgs> loss;
    std::vector<int> par(2 * n);
    int rc = RKG_OK;
    for (int m = 0; m < n && !rc; ++m) {
        rkg_grid* g = as[m]->g;
        if (g->speed_stale) rc = rkg_step(g, 0);   // make the control slot current
        d[m] = make_desc(g);
        if (as[m]->ng > 0) loss.push_back(loss_args(as[m]));
        par[m] = g->parity;
        par[n + m] = g->parity ^ 1;
    }
    if (rc) return rc;
    set_batch_tiles(n, as, d.data());
    for (int m = 0; m < n; ++m) batch_tiles(d[m], m, tiles);
    const size_t oT = al256(n * sizeof(GridDesc)), oL = oT + al256(tiles.size() * sizeof(BatchTile)),
                 oP = oL + al256((loss.size() + 1) * sizeof(LossArgs)), total = oP + al256(2 * n * sizeof(int));
    if (batch_tables(as[0], total)) return RKG_OK;
    ran = true;
    char *host = as[0]->batch_host, *dev = as[0]->batch_dev;
    std::memcpy(host, d.data(), n * sizeof(GridDesc));
    std::memcpy(host + oT, tiles.data(), tiles.size() * sizeof(BatchTile));
    if (!loss.empty()) std::memcpy(host + oL, loss.data(), loss.size() * sizeof(LossArgs));
    std::memcpy(host + oP, par.data(), 2 * n * sizeof(int));
    hipEvent_t join = nullptr;
    HIP_TRY(hipEventCreateWithFlags(&join, hipEventDisableTiming));
    hipError_t e = join_streams(n, as, join, true);
    if (e == hipSuccess) e = hipMemcpyAsync(dev, host, total, hipMemcpyHostToDevice, S);
    const GridDesc* dd = (const GridDesc*)dev;
    const BatchTile* dt = (const BatchTile*)(dev + oT);
    const dim3 grid((unsigned)tiles.size()), block(WAVE);
    for (int k = 0; k < nsteps && !rc && e == hipSuccess; ++k) {
        if (k % K == 0)
            for (int m = 0; m < n && !rc; ++m) rc = fwd_checkpoint(as[m], k / K, S);
        const int* dp = (const int*)(dev + oP) + (k & 1) * n;
        if (hllc) {
            hipLaunchKernelGGL((k_step_batch<1, true, false>), grid, block, 0, S, dd, dt, dp);
            hipLaunchKernelGGL((k_step_batch<2, true, false>), grid, block, 0, S, dd, dt, dp);
        } else {
            hipLaunchKernelGGL((k_step_batch<1, false, false>), grid, block, 0, S, dd, dt, dp);
            hipLaunchKernelGGL((k_step_batch<2, false, false>), grid, block, 0, S, dd, dt, dp);
        }
        for (int m = 0; m < n; ++m) as[m]->g->parity ^= 1;
        if (!loss.empty())
            hipLaunchKernelGGL(k_gauge_loss_batch, dim3((unsigned)loss.size()), dim3(256), 0, S,
                               (const LossArgs*)(dev + oL), k);
    }
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess) e = join_streams(n, as, join, false);
    // the tables may be rewritten once every launch that reads them has finished
    if (e != hipSuccess || rc) (void)hipStreamSynchronize(S);
    (void)hipEventDestroy(join);
    if (e != hipSuccess && !rc) { set_error("batched forward runs: %s", hipGetErrorString(e)); rc = RKG_ERR_HIP; }
    return rc;
}

// The reverse sweeps of n sessions as one sweep on the first session's
// stream: per replay step two launches (both stages of every member) and
// per reverse step eight (gauge seeds, the two stages' bodies and faces, the
// dt/clock kernels), each over the blocks of every member.  Every kernel
// argument of the whole sweep is known in advance (the sweep uses the first
// workspace set of every session) and is uploaded once.  The members'
// kernels and their block decompositions are those of their single-session
// sweeps, so each member's gradients are the same bits.  All sessions must
// use the same Riemann solver (HLL or HLLC).
int bwd_batched(int n, rkg_adjoint* const* as, double loss_scale) {
    const bool hllc = as[0]->g->cfg.use_hllc != 0;
    const int nsteps = as[0]->nsteps, K = as[0]->K, nseg = as[0]->nseg;
    std::vector<BwdPlan> pl(n);
    int rc = RKG_OK;
    // k_adj_y's rows too by the blocks of all members (us: 47 -> 41)
    long long yrows = 0;
    for (int m = 0; m < n; ++m) yrows += (long long)as[m]->g->cfg.ny * ((as[m]->g->cfg.nx + WAVE - 1) / WAVE);
    const int adj_rows = adj_y_rows(yrows);
    for (int m = 0; m < n && !rc; ++m) rc = bwd_begin(as[m], loss_scale, adj_rows, pl[m]);
    if (rc) return rc;
    for (int m = 0; m < n; ++m) use_set(as[m], 0);
    hipStream_t S = as[0]->g->stream;
    // every step's replay has the tiles of these
    std::vector<GridDesc> rec;
    for (int m = 0; m < n; ++m) rec.push_back(make_desc(as[m]->g));
    set_batch_tiles(n, as, rec.data());

    // block tables
    std::vector<BlockRef> tb, ty, tx, txr, tseed;
    std::vector<BatchTile> trec;
    for (int m = 0; m < n; ++m) {
        rkg_grid* g = as[m]->g;
        const int nx = g->cfg.nx, ny = g->cfg.ny;
        const int nb = pl[m].nb;
        for (int b = 0; b < nb; ++b) tb.push_back(BlockRef{m, b, nb, 0});
        const int yb = ((nx + WAVE - 1) / WAVE) * ((ny + pl[m].tile_rows - 1) / pl[m].tile_rows);
        for (int b = 0; b < yb; ++b) ty.push_back(BlockRef{m, b, yb, 0});
        // the edge strips of all members first (see adj_x)
        const int xb = x_blocks(nx, ny), xe = x_edge_blocks(nx, ny);
        for (int b = 0; b < xb; ++b) (b < xe ? tx : txr).push_back(BlockRef{m, b, xb, 0});
        if (as[m]->ng > 0) {
            const int sb = (as[m]->ncells + 255) / 256;
            for (int b = 0; b < sb; ++b) tseed.push_back(BlockRef{m, b, sb, 0});
        }
        batch_tiles(rec[m], m, trec);
    }
    tx.insert(tx.end(), txr.begin(), txr.end());
    // per global step: replay descriptors (stage 1, 2), replay parities, and
    // the reverse arguments (stage 2, stage 1, seeds, dt), n of each
    const size_t szGD = sizeof(GridDesc), szAS = sizeof(AdjStage), szSA = sizeof(SeedArgs), szDA = sizeof(DtArgs);
    auto al = [](size_t x) { return al256(x); };
    const size_t oRec1 = 0, oRec2 = oRec1 + al(n * szGD), oPar = oRec2 + al(n * szGD), oSt2 = oPar + al(n * sizeof(int)),
                 oSt1 = oSt2 + al(n * szAS), oSeed = oSt1 + al(n * szAS), oDt = oSeed + al(n * szSA),
                 step_bytes = oDt + al(n * szDA);
    const size_t tab_bytes = al(tb.size() * sizeof(BlockRef)) + al(ty.size() * sizeof(BlockRef)) +
                             al(tx.size() * sizeof(BlockRef)) + al(std::max<size_t>(1, tseed.size()) * sizeof(BlockRef)) +
                             al(trec.size() * sizeof(BatchTile));
    const size_t total = tab_bytes + step_bytes * (size_t)nsteps;
    if ((rc = batch_tables(as[0], total))) return rc;
    char *host = as[0]->batch_host, *dev = as[0]->batch_dev;
    hipEvent_t join = nullptr;
    HIP_TRY(hipEventCreateWithFlags(&join, hipEventDisableTiming));
    size_t off = 0;
    auto put = [&](const void* src, size_t bytes) {
        const size_t o = off;
        if (bytes) std::memcpy(host + o, src, bytes);
        off += al(bytes);
        return dev + o;
    };
    const BlockRef* dTb = (const BlockRef*)put(tb.data(), tb.size() * sizeof(BlockRef));
    const BlockRef* dTy = (const BlockRef*)put(ty.data(), ty.size() * sizeof(BlockRef));
    const BlockRef* dTx = (const BlockRef*)put(tx.data(), tx.size() * sizeof(BlockRef));
    const BlockRef* dTs = (const BlockRef*)put(tseed.data(), tseed.size() * sizeof(BlockRef));
    if (tseed.empty()) off += 256;
    const BatchTile* dTr = (const BatchTile*)put(trec.data(), trec.size() * sizeof(BatchTile));
    off = tab_bytes;
    for (int s = 0; s < nseg; ++s) {
        for (int k = 0; k < seg_steps(as[0], s); ++k) {
            char* h = host + tab_bytes + step_bytes * (size_t)(s * K + k);
            for (int m = 0; m < n; ++m) {
                rkg_adjoint* a = as[m];
                GridDesc d1 = stage_desc(a, wsA(a, k), wsB(a, k), wsA(a, k + 1));
                copy_tiles(d1, rec[m]);
                d1.rec = wsD1(a, k);
                d1.hist = a->hist + HIST * k;
                GridDesc d2 = d1;
                d2.rec = wsD2(a, k);
                d2.hist = nullptr;
                std::memcpy(h + oRec1 + m * szGD, &d1, szGD);
                std::memcpy(h + oRec2 + m * szGD, &d2, szGD);
                const int par = a->ckpt_parity[s] ^ (k & 1);
                std::memcpy(h + oPar + m * sizeof(int), &par, sizeof(int));
                const AdjStage st2 = stage_args(a, k, 2, pl[m]);
                const AdjStage st1 = stage_args(a, k, 1, pl[m]);
                const SeedArgs sa = seed_args(a, k, s * K + k, pl[m]);
                const DtArgs da = dt_args(a, k, st1, pl[m]);
                std::memcpy(h + oSt2 + m * szAS, &st2, szAS);
                std::memcpy(h + oSt1 + m * szAS, &st1, szAS);
                std::memcpy(h + oSeed + m * szSA, &sa, szSA);
                std::memcpy(h + oDt + m * szDA, &da, szDA);
            }
        }
    }
    // the sweep starts after every member's queued work (bwd_begin's clears)
    hipError_t e = join_streams(n, as, join, true);
    if (e == hipSuccess) e = hipMemcpyAsync(dev, host, total, hipMemcpyHostToDevice, S);
    if (e != hipSuccess) {
        (void)hipEventDestroy(join);
        set_error("batched adjoint sweep: %s", hipGetErrorString(e));
        return RKG_ERR_HIP;
    }
    const int nrec = (int)trec.size();
    for (int s = nseg - 1; s >= 0 && !rc; --s) {
        for (int m = 0; m < n && !rc; ++m) rc = bwd_replay_begin(as[m], s, pl[m], S);
        if (rc) break;
        const int Ks = seg_steps(as[0], s);
        for (int k = 0; k < Ks; ++k) {
            const char* d = dev + tab_bytes + step_bytes * (size_t)(s * K + k);
            const GridDesc* r1 = (const GridDesc*)(d + oRec1);
            const GridDesc* r2 = (const GridDesc*)(d + oRec2);
            const int* par = (const int*)(d + oPar);
            if (hllc) {
                hipLaunchKernelGGL((k_step_batch<1, true, true>), dim3(nrec), dim3(WAVE), 0, S, r1, dTr, par);
                hipLaunchKernelGGL((k_step_batch<2, true, true>), dim3(nrec), dim3(WAVE), 0, S, r2, dTr, par);
            } else {
                hipLaunchKernelGGL((k_step_batch<1, false, true>), dim3(nrec), dim3(WAVE), 0, S, r1, dTr, par);
                hipLaunchKernelGGL((k_step_batch<2, false, true>), dim3(nrec), dim3(WAVE), 0, S, r2, dTr, par);
            }
        }
        for (int k = Ks - 1; k >= 0; --k) {
            const char* d = dev + tab_bytes + step_bytes * (size_t)(s * K + k);
            const AdjStage* st2 = (const AdjStage*)(d + oSt2);
            const AdjStage* st1 = (const AdjStage*)(d + oSt1);
            if (!tseed.empty())
                hipLaunchKernelGGL(k_gauge_seed_batch, dim3((int)tseed.size()), dim3(256), 0, S,
                                   (const SeedArgs*)(d + oSeed), dTs);
            hipLaunchKernelGGL(k_adj_body_batch<2>, dim3((int)tb.size()), dim3(256), 0, S, st2, dTb);
            if (hllc) {
                hipLaunchKernelGGL((k_adj_y_batch<true, 2>), dim3((int)ty.size()), dim3(WAVE), 0, S, st2, dTy);
                hipLaunchKernelGGL((k_adj_x_batch<true, 2>), dim3((int)tx.size()), dim3(WAVE), 0, S, st2, dTx);
            } else {
                hipLaunchKernelGGL((k_adj_y_batch<false, 2>), dim3((int)ty.size()), dim3(WAVE), 0, S, st2, dTy);
                hipLaunchKernelGGL((k_adj_x_batch<false, 2>), dim3((int)tx.size()), dim3(WAVE), 0, S, st2, dTx);
            }
            hipLaunchKernelGGL(k_adj_body_batch<1>, dim3((int)tb.size()), dim3(256), 0, S, st1, dTb);
            if (hllc) {
                hipLaunchKernelGGL((k_adj_y_batch<true, 1>), dim3((int)ty.size()), dim3(WAVE), 0, S, st1, dTy);
                hipLaunchKernelGGL((k_adj_x_batch<true, 1>), dim3((int)tx.size()), dim3(WAVE), 0, S, st1, dTx);
            } else {
                hipLaunchKernelGGL((k_adj_y_batch<false, 1>), dim3((int)ty.size()), dim3(WAVE), 0, S, st1, dTy);
                hipLaunchKernelGGL((k_adj_x_batch<false, 1>), dim3((int)tx.size()), dim3(WAVE), 0, S, st1, dTx);
            }
            hipLaunchKernelGGL(k_dt_rev_batch, dim3(n), dim3(1024), 0, S, (const DtArgs*)(d + oDt));
        }
    }
    if (!rc) e = hipGetLastError();
    // every member's stream continues after the sweep
    if (!rc && e == hipSuccess) e = join_streams(n, as, join, false);
    if (!rc && e != hipSuccess) { set_error("batched adjoint sweep: %s", hipGetErrorString(e)); rc = RKG_ERR_HIP; }
    for (int m = 0; m < n && !rc; ++m) rc = bwd_end(as[m]);
    // the tables may be rewritten once every launch that reads them has finished
    for (int m = 0; m < n; ++m) (void)hipStreamSynchronize(as[m]->g->stream);
    (void)hipEventDestroy(join);
    trim_tables(as[0]);
    if (rc) return rc;
    for (int m = 0; m < n && !rc; ++m) rc = bwd_finish(as[m]);
    return rc;
}

// Sessions of one batch: valid, distinct grids on distinct streams, with
// one step count and checkpoint interval.
int check_batch(int n, rkg_adjoint* const* as) {
    if (n < 1 || !as) { set_error("need at least one session"); return RKG_ERR_RANGE; }
    for (int m = 0; m < n; ++m) {
        if (!valid(as[m])) return RKG_ERR_BAD_HANDLE;
        if (as[m]->nsteps != as[0]->nsteps || as[m]->K != as[0]->K) {
            set_error("sessions of a batch need the same step count and checkpoint interval");
            return RKG_ERR_RANGE;
        }
        for (int q = 0; q < m; ++q)
            if (as[q]->g == as[m]->g || as[q]->g->stream == as[m]->g->stream) {
                set_error("sessions %d and %d share a grid or a stream", q, m);
                return RKG_ERR_RANGE;
            }
    }
    return RKG_OK;
}

}  // namespace

extern "C" {

// nsteps steps from the grid's current state, recording checkpoints and the
// gauge misfit; the grid is left at the final state.
int rkg_adjoint_forward(rkg_adjoint* a, double* loss) {
    if (!valid(a)) return RKG_ERR_BAD_HANDLE;
    int rc = fwd_begin(a);
    for (int n = 0; !rc && n < a->nsteps; ++n) rc = fwd_step(a, n);
    if (!rc) rc = fwd_end(a);
    if (rc) return rc;
    HIP_TRY(hipStreamSynchronize(a->g->stream));
    return fwd_finish(a, loss);
}

// Reverse sweep: gradients of loss_scale * L with respect to the bed, the
// per-cell Manning n and the initial state (h, hu, hv).  The grid's state
// is left as the forward run left it.
int rkg_adjoint_backward(rkg_adjoint* a, double loss_scale, int tile_rows) {
    if (!valid(a)) return RKG_ERR_BAD_HANDLE;
    if (!a->have_forward) { set_error("rkg_adjoint_backward before rkg_adjoint_forward"); return RKG_ERR_NOT_READY; }
    ensure_overlap(a);   // before the sweep's start event: the first call allocates
    BwdPlan pl;
    int rc = bwd_begin(a, loss_scale, tile_rows, pl);
    if (rc) return rc;
    if (a->rstream) {
        rc = bwd_overlapped(a, pl);
    } else {
        for (int s = a->nseg - 1; s >= 0 && !rc; --s) {
            rc = bwd_replay_begin(a, s, pl, a->g->stream);
            if (rc) break;
            for (int k = 0; k < seg_steps(a, s); ++k) bwd_replay_step(a, k, pl, a->g->stream);
            for (int k = seg_steps(a, s) - 1; k >= 0; --k) bwd_reverse_step(a, s, k, pl);
        }
    }
    if (rc) return rc;
    rc = bwd_end(a);
    if (rc) return rc;
    HIP_TRY(hipStreamSynchronize(a->g->stream));
    return bwd_finish(a);
}

// The forward runs of n sessions (one grid and stream each): as one run
// where they can (fwd_batchable), else queued step by step across the
// sessions so that their kernels overlap.
int rkg_adjoint_forward_many(int n, rkg_adjoint* const* as, double* losses) {
    int rc = check_batch(n, as);
    if (rc) return rc;
    for (int m = 0; m < n && !rc; ++m) rc = fwd_begin(as[m]);
    bool ran = false;
    if (!rc && fwd_batchable(n, as)) rc = fwd_batched(n, as, ran);
    for (int k = 0; k < as[0]->nsteps && !rc && !ran; ++k)
        for (int m = 0; m < n && !rc; ++m) rc = fwd_step(as[m], k);
    for (int m = 0; m < n && !rc; ++m) rc = fwd_end(as[m]);
    if (rc) return rc;
    for (int m = 0; m < n; ++m) HIP_TRY(hipStreamSynchronize(as[m]->g->stream));
    trim_tables(as[0]);
    for (int m = 0; m < n && !rc; ++m) rc = fwd_finish(as[m], losses ? losses + m : nullptr);
    return rc;
}

// The reverse sweeps of n sessions, queued step by step across the
// sessions (replays, then reverse steps, segment by segment).  Each
// session's gradients are those of rkg_adjoint_backward.
int rkg_adjoint_backward_many(int n, rkg_adjoint* const* as, double loss_scale) {
    int rc = check_batch(n, as);
    if (rc) return rc;
    bool same_solver = true;
    for (int m = 1; m < n; ++m) same_solver = same_solver && as[m]->g->cfg.use_hllc == as[0]->g->cfg.use_hllc;
    if (same_solver) return bwd_batched(n, as, loss_scale);
    // sessions mixing HLL and HLLC: their own kernels, interleaved on their streams
    std::vector<BwdPlan> pl(n);
    for (int m = 0; m < n && !rc; ++m) rc = bwd_begin(as[m], loss_scale, 0, pl[m]);
    for (int s = as[0]->nseg - 1; s >= 0 && !rc; --s) {
        for (int m = 0; m < n && !rc; ++m) rc = bwd_replay_begin(as[m], s, pl[m], as[m]->g->stream);
        if (rc) break;
        const int Ks = seg_steps(as[0], s);
        for (int k = 0; k < Ks; ++k)
            for (int m = 0; m < n; ++m) bwd_replay_step(as[m], k, pl[m], as[m]->g->stream);
        for (int k = Ks - 1; k >= 0; --k)
            for (int m = 0; m < n; ++m) bwd_reverse_step(as[m], s, k, pl[m]);
    }
    for (int m = 0; m < n && !rc; ++m) rc = bwd_end(as[m]);
    if (rc) return rc;
    for (int m = 0; m < n; ++m) HIP_TRY(hipStreamSynchronize(as[m]->g->stream));
    for (int m = 0; m < n && !rc; ++m) rc = bwd_finish(as[m]);
    return rc;
}

// Adds the adjoint of a still-water initial state (h = max(eta0 - b, 0),
// hu = hv = 0) to the bed gradient.
int rkg_adjoint_fold_still_water(rkg_adjoint* a, double eta0) {
    if (!valid(a)) return RKG_ERR_BAD_HANDLE;
    rkg_grid* g = a->g;
    hipLaunchKernelGGL(k_fold_still_water, dim3(body_blocks(g)), dim3(256), 0, g->stream, g->buf + 6 * g->plane,
                       lamA(a), eta0, g->cfg.nx, g->cfg.ny, (long long)g->pitch, gradB(a));
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(g->stream));
    return RKG_OK;
}

// field: RKG_FIELD_B (bed), RKG_FIELD_N (Manning n), RKG_FIELD_H/HU/HV
// (initial state).  on_device != 0: dst is device memory.
int rkg_adjoint_gradient(rkg_adjoint* a, int field, double* dst, int ld, int on_device) {
    if (!valid(a)) return RKG_ERR_BAD_HANDLE;
    rkg_grid* g = a->g;
    const double* src;
    switch (field) {
    case RKG_FIELD_H: src = lamA(a); break;
    case RKG_FIELD_HU: src = lamA(a) + g->plane; break;
    case RKG_FIELD_HV: src = lamA(a) + 2 * g->plane; break;
    case RKG_FIELD_B: src = gradB(a); break;
    case RKG_FIELD_N: src = gradN(a); break;
    default: set_error("no gradient for field %d", field); return RKG_ERR_RANGE;
    }
    if (!dst || ld < g->cfg.nx) { set_error("bad buffer or leading dimension"); return RKG_ERR_RANGE; }
    const size_t W = sizeof(double), nx = (size_t)g->cfg.nx, ny = (size_t)g->cfg.ny, pitch = (size_t)g->pitch;
    if (!on_device) {
        HIP_TRY(plane_to_host(*g->stage, dst, (size_t)ld, src, pitch, nx, ny, g->stream));
        return RKG_OK;
    }
    HIP_TRY(hipMemcpy2DAsync(dst, (size_t)ld * W, src, pitch * W, nx * W, ny, hipMemcpyDeviceToDevice, g->stream));
    HIP_TRY(hipStreamSynchronize(g->stream));
    return RKG_OK;
}

int rkg_adjoint_timing(rkg_adjoint* a, double* forward_ms, double* backward_ms) {
    if (!valid(a)) return RKG_ERR_BAD_HANDLE;
    if (forward_ms) *forward_ms = a->fwd_ms;
    if (backward_ms) *backward_ms = a->bwd_ms;
    return RKG_OK;
}

}  // extern "C"
