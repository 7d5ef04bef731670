// swe_core.hpp -- per-face and per-cell arithmetic of the structured 2-D
// shallow-water step, as gfx950 device functions.
//
// The step is Rakali's SSP-RK2 barotropic step (rki_solver.F90:761-815):
// Audusse hydrostatic reconstruction with minmod MUSCL slopes, HLL/HLLC
// Riemann fluxes with Ritter dry-front speeds, the well-balanced pressure
// correction, and the fused Euler update with clamp, KP07
// desingularization, Froude backstop, semi-implicit Manning and Coriolis.
//
// Arithmetic is written expression-for-expression in the reference's
// evaluation order and built with -ffp-contract=off, so each face and cell
// value is the IEEE result of the same operation sequence.  The reference
// evaluates every interior face twice (once from each cell,
// rki_kernel_flux.F90:371-372) and both evaluations are bit-identical,
// because a face depends only on the four cells across it; here each
// cell's slopes are evaluated once (cell_states) and each face once
// (face_flux), and the face is handed to both of its cells.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cstring>

#include "crmath.hpp"

namespace rk {

// rki_constants.F90:53,59,68-73,120
constexpr double DRY_TOLERANCE = 1.0e-6;
constexpr double THIN_LAYER_THRESHOLD = 1.0e-3;
constexpr double DESING_EPS = 1.5e-4;
constexpr double FROUDE_BACKSTOP = 50.0;
constexpr double RHO_WATER = 1035.0;          // rki_constants.F90:40
constexpr double TWO_PI = 6.283185307179586;  // 8*atan(1), rki_constants.F90:114
constexpr double SQRT2 = 1.4142135623730951;  // sqrt(2.0_wp) folded

// Boundary tags (rki_boundary_types.F90:18-32).
enum : int { BC_WALL = 1, BC_OPEN = 2, BC_TIDAL = 3, BC_NESTED = 4, BC_INFLOW = 5,
             BC_DISCHARGE = 6, BC_CLAMPED = 7, BC_SPONGE = 8, BC_CHAPMAN = 9 };

struct Cell {
    double h, hu, hv, b;
};

// One face's contribution to its two cells.  a = h_hyd_r^2 - h_R^2 is the
// right cell's "left" pressure term; c = h_hyd_l^2 and d = h_L^2 are the
// left cell's "right" terms (rki_kernel_flux.F90:361-369 evaluates
// ((hyd_left^2 - pre_left^2) - hyd_right^2) + pre_right^2).
struct Face {
    double fh, fhu, fhv, a, c, d;
};

__host__ __device__ __forceinline__ double fmax0(double x) { return x > 0.0 ? x : 0.0; }
__host__ __device__ __forceinline__ double dmax(double a, double b) { return a > b ? a : b; }
__host__ __device__ __forceinline__ double dmin(double a, double b) { return a < b ? a : b; }
// x**4 as LLVM flang lowers it for a run-time base: ((x*x)*x)*x.
__device__ __forceinline__ double pow4(double x) { return ((x * x) * x) * x; }

// IEEE division by a denominator shared between several numerators.
// The compiler's f64 division is v_div_scale (identity for operands away
// from the exponent extremes), v_rcp, two Newton refinements of the
// reciprocal, a product, a residual fma and the correction fma
// (v_div_fmas), then v_div_fixup (identity for finite, non-zero operands).
// Recip keeps the refined reciprocal, so each further quotient by the same
// denominator costs a product and two fmas and returns the same bits as
// `n / d`.  The residual is formed as -fma(d, q0, -n) so that zero
// numerators keep their sign.  Two Newton steps, as the division takes.  One cubic
// step from v_rcp is an fma less, but leaves 1 / d within 2^-72 before its rounding
// and so the wrong one of two doubles where 1 / d lies that close to the middle
// between them: 113 of the 9e6 operands that can tell gave another quotient than
// the division then (tests/quotients.hip enumerates them).  (The division itself
// misrounds three of them, all with d of the form 2^k (1 - 5, 11 or 13 2^-53).)
// The unscaled sequence equals the IEEE quotient while |n| >= 2^-969 (or n = 0)
// and the denominator is far from the exponent extremes; callers guarantee the
// numerator bound by running a row with EXACT = true (plain division) whenever a
// cell of its stencil holds a value that is unbounded().
struct Recip {
    double d, y;
};

__device__ __forceinline__ Recip recip(double d) {
    const double y0 = __builtin_amdgcn_rcp(d);
    const double y1 = fma(y0, fma(-d, y0, 1.0), y0);
    return Recip{d, fma(y1, fma(-d, y1, 1.0), y1)};
}

template <bool EXACT>
__device__ __forceinline__ double rdiv(double n, const Recip& r) {
    if (EXACT) return n / r.d;
    const double q0 = n * r.y;
    const double t = fma(r.d, q0, -n);
    return fma(-t, r.y, q0);
}

// Division by a grid spacing.  Where the spacing has at most 50 significant
// bits (`two_op`; 10, 20, 62.5 and the like), the quotient is
// fma(n, yh, n yl) with 1/d = yh + yl: the value before its rounding is
// within 2^-52 ulp of n / d, and such a quotient is at least 2^-51 ulp from
// every rounding boundary (n 2^t - odd D is a non-zero integer, over D <
// 2^50), so the result is the IEEE quotient at two operations instead of
// three.  Another spacing takes rdiv.
struct Spacing {
    Recip r;
    double yl;
    bool two_op;
};

inline Spacing spacing(double d) {   // on the host, once per launch
    Spacing s;
    uint64_t u;
    memcpy(&u, &d, sizeof u);
    s.r.d = d;
    s.r.y = 1.0 / d;
    s.yl = __builtin_fma(-d, s.r.y, 1.0) * s.r.y;   // the residual is exact
    s.two_op = (u & 7) == 0;
    return s;
}

template <bool TWO>
__device__ __forceinline__ double sdiv(double n, const Spacing& s) {
    return TWO ? fma(n, s.r.y, n * s.yl) : rdiv<false>(n, s.r);
}

// A depth or momentum that is non-zero and outside [2^-300, 2^40] in
// magnitude, or a bed above 2^40, or a value that is not finite: one for which
// some quotient of the step could leave the range where rdiv<false> is
// exact, or another range argument of the row path (below) does not hold.  (A
// tiny bed next to ordinary depths changes none of them.)
__device__ __forceinline__ bool unbounded(double x) {
    const double a = fabs(x);
    return (x != 0.0) & !((a >= 0x1p-300) & (a <= 0x1p40));
}

// Square root of a finite x >= 2^-767: the correctly rounded sequence the
// compiler emits for sqrt (reciprocal square root, Goldschmidt refinement,
// two fma residual corrections) without its scaling of inputs below
// 2^-767 and its fixup of 0 and infinity, which are identities on that
// range.  Same bits as sqrt(x) there.
__device__ __forceinline__ double sqrt_pos(double x) {
    const double r = __builtin_amdgcn_rsq(x);
    double g = x * r;
    double h = r * 0.5;
    const double e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    double d = fma(-g, g, x);
    g = fma(d, h, g);
    d = fma(-g, g, x);
    return fma(d, h, g);
}
__device__ __forceinline__ bool unbounded(const Cell& c) {
    return unbounded(c.h) | unbounded(c.hu) | unbounded(c.hv) | !(fabs(c.b) <= 0x1p40);
}

// minmod, rki_kernel_flux.F90:380-393
__device__ __forceinline__ double minmod(double a, double b) {
    if (a * b <= 0.0) return 0.0;
    return (fabs(a) < fabs(b)) ? a : b;
}

// HLL / HLLC normal flux in x: rki_kernel_flux.F90:410-495 and 584-684.
template <bool HLLC>
__device__ __forceinline__ void riemann_x(double g, double h_l, double hu_l, double hv_l,
                                          double h_r, double hu_r, double hv_r,
                                          double& f_h, double& f_hu, double& f_hv) {
    double u_l = 0.0, v_l = 0.0, u_r = 0.0, v_r = 0.0;
    if (h_l > DRY_TOLERANCE) { u_l = hu_l / h_l; v_l = hv_l / h_l; }
    if (h_r > DRY_TOLERANCE) { u_r = hu_r / h_r; v_r = hv_r / h_r; }
    const double a_l = sqrt(g * fmax0(h_l));
    const double a_r = sqrt(g * fmax0(h_r));
    double s_l, s_r;
    if (h_r <= DRY_TOLERANCE) {          // dry right: Ritter front speed
        s_l = u_l - a_l;
        s_r = u_l + 2.0 * a_l;
    } else if (h_l <= DRY_TOLERANCE) {   // dry left
        s_l = u_r - 2.0 * a_r;
        s_r = u_r + a_r;
    } else {                             // Davis
        s_l = dmin(u_l - a_l, u_r - a_r);
        s_r = dmax(u_l + a_l, u_r + a_r);
    }
    const double fl_h = hu_l, fl_hu = hu_l * u_l + 0.5 * g * h_l * h_l, fl_hv = hu_l * v_l;
    const double fr_h = hu_r, fr_hu = hu_r * u_r + 0.5 * g * h_r * h_r, fr_hv = hu_r * v_r;
    if (s_l >= 0.0) {
        f_h = fl_h; f_hu = fl_hu; f_hv = fl_hv;
    } else if (s_r <= 0.0) {
        f_h = fr_h; f_hu = fr_hu; f_hv = fr_hv;
    } else {
        const double denom = 1.0 / (s_r - s_l);
        f_h = (s_r * fl_h - s_l * fr_h + s_l * s_r * (h_r - h_l)) * denom;
        f_hu = (s_r * fl_hu - s_l * fr_hu + s_l * s_r * (hu_r - hu_l)) * denom;
        if (!HLLC) {
            f_hv = (s_r * fl_hv - s_l * fr_hv + s_l * s_r * (hv_r - hv_l)) * denom;
        } else {
            // contact speed, rki_kernel_flux.F90:670-681
            const double denom_star = h_r * (u_r - s_r) - h_l * (u_l - s_l);
            double s_star;
            if (fabs(denom_star) > DRY_TOLERANCE)
                s_star = (s_l * h_r * (u_r - s_r) - s_r * h_l * (u_l - s_l)) / denom_star;
            else
                s_star = 0.5 * (u_l + u_r);
            f_hv = (s_star >= 0.0) ? f_h * v_l : f_h * v_r;
        }
    }
}

// HLL / HLLC normal flux in y: rki_kernel_flux.F90:497-582 and 686-783.
// Arguments are (h, hu, hv) of the bottom then the top state, as there.
template <bool HLLC>
__device__ __forceinline__ void riemann_y(double g, double h_b, double hu_b, double hv_b,
                                          double h_t, double hu_t, double hv_t,
                                          double& g_h, double& g_hu, double& g_hv) {
    double u_b = 0.0, v_b = 0.0, u_t = 0.0, v_t = 0.0;
    if (h_b > DRY_TOLERANCE) { u_b = hu_b / h_b; v_b = hv_b / h_b; }
    if (h_t > DRY_TOLERANCE) { u_t = hu_t / h_t; v_t = hv_t / h_t; }
    const double a_b = sqrt(g * fmax0(h_b));
    const double a_t = sqrt(g * fmax0(h_t));
    double s_l, s_r;
    if (h_t <= DRY_TOLERANCE) {
        s_l = v_b - a_b;
        s_r = v_b + 2.0 * a_b;
    } else if (h_b <= DRY_TOLERANCE) {
        s_l = v_t - 2.0 * a_t;
        s_r = v_t + a_t;
    } else {
        s_l = dmin(v_b - a_b, v_t - a_t);
        s_r = dmax(v_b + a_b, v_t + a_t);
    }
    const double gl_h = hv_b, gl_hu = hu_b * v_b, gl_hv = hv_b * v_b + 0.5 * g * h_b * h_b;
    const double gr_h = hv_t, gr_hu = hu_t * v_t, gr_hv = hv_t * v_t + 0.5 * g * h_t * h_t;
    if (s_l >= 0.0) {
        g_h = gl_h; g_hu = gl_hu; g_hv = gl_hv;
    } else if (s_r <= 0.0) {
        g_h = gr_h; g_hu = gr_hu; g_hv = gr_hv;
    } else {
        const double denom = 1.0 / (s_r - s_l);
        g_h = (s_r * gl_h - s_l * gr_h + s_l * s_r * (h_t - h_b)) * denom;
        g_hv = (s_r * gl_hv - s_l * gr_hv + s_l * s_r * (hv_t - hv_b)) * denom;
        if (!HLLC) {
            g_hu = (s_r * gl_hu - s_l * gr_hu + s_l * s_r * (hu_t - hu_b)) * denom;
        } else {
            const double denom_star = h_t * (v_t - s_r) - h_b * (v_b - s_l);
            double s_star;
            if (fabs(denom_star) > DRY_TOLERANCE)
                s_star = (s_l * h_t * (v_t - s_r) - s_r * h_b * (v_b - s_l)) / denom_star;
            else
                s_star = 0.5 * (v_b + v_t);
            g_hu = (s_star >= 0.0) ? g_h * u_b : g_h * u_t;
        }
    }
}

// Reconstructed state of a cell at one of its faces along a direction:
// h = max(0, eta_face - b) and the reconstructed momenta (the bed is the
// cell's own).
struct FState {
    double h, hu, hv;
};

// Minmod-limited MUSCL states of cell c at its low (lo) and high (hi) face
// along one direction, from its neighbours m (below) and p (above):
// rki_kernel_flux.F90:158-181 for the slope (zeroed near wet/dry fronts),
// :186-189 / :229-232 for the face states.  Each face of the reference
// re-evaluates this slope for both of its cells; a cell's slope is the
// same from both of its faces, so it is evaluated once here.
__device__ __forceinline__ void cell_states(const Cell& m, const Cell& c, const Cell& p, FState& lo,
                                            FState& hi) {
    const double e_m = m.h + m.b;
    const double e_c = c.h + c.b;
    const double e_p = p.h + p.b;
    double s_eta, s_hu, s_hv;
    if (c.h < THIN_LAYER_THRESHOLD || m.h < DRY_TOLERANCE || p.h < DRY_TOLERANCE) {
        s_eta = 0.0; s_hu = 0.0; s_hv = 0.0;
    } else {
        s_eta = minmod(e_c - e_m, e_p - e_c);
        s_hu = minmod(c.hu - m.hu, p.hu - c.hu);
        s_hv = minmod(c.hv - m.hv, p.hv - c.hv);
    }
    lo.h = fmax0((e_c - 0.5 * s_eta) - c.b);
    lo.hu = c.hu - 0.5 * s_hu;
    lo.hv = c.hv - 0.5 * s_hv;
    hi.h = fmax0((e_c + 0.5 * s_eta) - c.b);
    hi.hu = c.hu + 0.5 * s_hu;
    hi.hv = c.hv + 0.5 * s_hv;
}

// One face between the high state L of its left cell (bed bL) and the low
// state R of its right cell (bed bR): Audusse hydrostatic reconstruction
// (rki_kernel_flux.F90:208-210), velocities (extract_velocity, :395-408)
// and the HLL/HLLC flux of the h_hyd-weighted momenta (:216-224).
template <bool HLLC, bool YDIR>
__device__ __forceinline__ Face face_flux(double g, const FState& L, double bL, const FState& R,
                                          double bR) {
    const double b_max = dmax(bL, bR);
    const double h_hyd_l = fmax0(L.h + bL - b_max);
    const double h_hyd_r = fmax0(R.h + bR - b_max);
    double u_l = 0.0, v_l = 0.0, u_r = 0.0, v_r = 0.0;
    if (L.h > DRY_TOLERANCE) { u_l = L.hu / L.h; v_l = L.hv / L.h; }
    if (R.h > DRY_TOLERANCE) { u_r = R.hu / R.h; v_r = R.hv / R.h; }
    Face f;
    if (YDIR)
        riemann_y<HLLC>(g, h_hyd_l, h_hyd_l * u_l, h_hyd_l * v_l, h_hyd_r, h_hyd_r * u_r,
                        h_hyd_r * v_r, f.fh, f.fhu, f.fhv);
    else
        riemann_x<HLLC>(g, h_hyd_l, h_hyd_l * u_l, h_hyd_l * v_l, h_hyd_r, h_hyd_r * u_r,
                        h_hyd_r * v_r, f.fh, f.fhu, f.fhv);
    f.a = h_hyd_r * h_hyd_r - R.h * R.h;
    f.c = h_hyd_l * h_hyd_l;
    f.d = L.h * L.h;
    return f;
}

// ---------------------------------------------------------------------
// The row path.  Every row whose stencil passes unbounded() is evaluated by
// the functions below (states_row, face_row, stage_body_row, ...); the
// functions above, with plain divisions, take the others.  Both perform the
// same rounded operations on every value that is used, so the bits do not
// depend on the path.  The row path is written for a wavefront that is
// bound by instruction issue (about 0.65 of the issue slots, three waves per
// SIMD): branches are selects, and selects are few:
//  * max(x, 0), max(a, b) and minmod are v_max_f64 / v_min_f64 (one
//    instruction instead of a compare and two selects).  They differ from
//    the compare-and-select forms only in the sign of a zero;
//  * minmod(a, b) = max(min(a, b), 0) + min(max(a, b), 0): one of the two
//    terms is the limited slope and the other is zero.  The reference zeroes
//    the slope where a b <= 0; a and b are differences of values that are 0
//    or at least 2^-300, hence 0 or at least 2^-352, and a b does not
//    underflow;
//  * c -+ 0.5 s is one fma: 0.5 s is exact.  Where the slopes are zeroed the
//    factor 0.5 becomes 0, one select for the three slopes;
//  * a dry side's velocities are zeroed through its reciprocal (n * 0), one
//    select for both quotients.  A wavefront whose faces are wet takes a copy
//    of the face without these selects;
//  * square roots of g h take sqrt_pos: with h 0 or at least 2^-353 (a
//    difference of bounded values) the argument is 0, where the result is
//    selected, or above 2^-767;
//  * 1 / (s_r - s_l) is a shared-reciprocal quotient: in the star region the
//    span is at least 2^-180 and at most 2^45, far from the exponents where
//    the division would scale;
//  * HLLC needs only the sign of s_star.  In the star region u_r - s_r <= 0
//    and u_l - s_l >= 0 (Davis or Ritter speeds), so denom_star <= 0 and
//    s_star >= 0 where num <= 0.  With denom_star < -DRY_TOLERANCE a non-zero
//    num is a rounded difference of terms whose larger one is at least 2^-89
//    (|s| >= 2^-68 where a side has h > DRY_TOLERANCE and g >= 1e-3, depth
//    times relative speed at least 2^-21), so |num| >= 2^-142; and
//    |denom_star| is below 2^83: the quotient does not underflow.

__device__ __forceinline__ double vmax(double a, double b) { return __builtin_fmax(a, b); }
__device__ __forceinline__ double vmin(double a, double b) { return __builtin_fmin(a, b); }
__device__ __forceinline__ double minmod_row(double a, double b) {
    return vmax(vmin(a, b), 0.0) + vmin(vmax(a, b), 0.0);
}

// cell_states from the surface and momenta (e, hu, hv) of the three cells and
// the bed of the middle one; `flat` where the slopes are zeroed.
struct Surf {
    double e, hu, hv;
};
__device__ __forceinline__ Surf operator-(const Surf& a, const Surf& b) {
    return Surf{a.e - b.e, a.hu - b.hu, a.hv - b.hv};
}
__device__ __forceinline__ void states_row(const Surf& dm, const Surf& dp, const Surf& c, double b, bool flat,
                                           FState& lo, FState& hi) {
    const double w = flat ? 0.0 : 0.5;
    const double s_eta = minmod_row(dm.e, dp.e);
    const double s_hu = minmod_row(dm.hu, dp.hu);
    const double s_hv = minmod_row(dm.hv, dp.hv);
    lo.h = vmax(fma(-w, s_eta, c.e) - b, 0.0);
    lo.hu = fma(-w, s_hu, c.hu);
    lo.hv = fma(-w, s_hv, c.hv);
    hi.h = vmax(fma(w, s_eta, c.e) - b, 0.0);
    hi.hu = fma(w, s_hu, c.hu);
    hi.hv = fma(w, s_hv, c.hv);
}

// face_flux of the row path.  DRY: some lane that matters has a dry side
// (or hydrostatic depth); without it all four depths are wet.
template <bool HLLC, bool YDIR, bool DRY>
__device__ __forceinline__ Face face_row_as(double g, const FState& L, const FState& R, double h_l, double h_r,
                                            bool use) {
    Recip rL = recip(L.h), rR = recip(R.h), rl = recip(h_l), rr = recip(h_r);
    const bool dry_l = h_l <= DRY_TOLERANCE, dry_r = h_r <= DRY_TOLERANCE;
    if (DRY) {
        rL.y = L.h > DRY_TOLERANCE ? rL.y : 0.0;
        rR.y = R.h > DRY_TOLERANCE ? rR.y : 0.0;
        rl.y = dry_l ? 0.0 : rl.y;
        rr.y = dry_r ? 0.0 : rr.y;
    }
    const double q0_l = h_l * rdiv<false>(L.hu, rL), q1_l = h_l * rdiv<false>(L.hv, rL);
    const double q0_r = h_r * rdiv<false>(R.hu, rR), q1_r = h_r * rdiv<false>(R.hv, rR);
    // normal and tangential momentum of the hydrostatic states
    const double n_l = YDIR ? q1_l : q0_l, t_l = YDIR ? q0_l : q1_l;
    const double n_r = YDIR ? q1_r : q0_r, t_r = YDIR ? q0_r : q1_r;
    const double u_l = rdiv<false>(n_l, rl), v_l = rdiv<false>(t_l, rl);
    const double u_r = rdiv<false>(n_r, rr), v_r = rdiv<false>(t_r, rr);
    double a_l = sqrt_pos(g * h_l), a_r = sqrt_pos(g * h_r);
    if (DRY) {
        a_l = h_l > 0.0 ? a_l : 0.0;
        a_r = h_r > 0.0 ? a_r : 0.0;
    }
    double s_l = vmin(u_l - a_l, u_r - a_r);
    double s_r = vmax(u_l + a_l, u_r + a_r);
    if (DRY) {   // Ritter fronts
        s_l = dry_r ? u_l - a_l : (dry_l ? fma(-2.0, a_r, u_r) : s_l);
        s_r = dry_r ? fma(2.0, a_l, u_l) : (dry_l ? u_r + a_r : s_r);
    }
    const double half_g = 0.5 * g;
    // x faces: fl_hv = hu_l v_l; y faces: gl_hu = hu_b v_b (the operand order of the reference)
    const double fl_n = n_l * u_l + half_g * h_l * h_l, fr_n = n_r * u_r + half_g * h_r * h_r;
    const double denom = rdiv<false>(1.0, recip(s_r - s_l));
    const double ss = s_l * s_r;
    Face f;
    double fn, ft;
    f.fh = (s_r * n_l - s_l * n_r + ss * (h_r - h_l)) * denom;
    fn = (s_r * fl_n - s_l * fr_n + ss * (n_r - n_l)) * denom;
    double fl_t = 0.0, fr_t = 0.0;
    if (!HLLC) {
        fl_t = YDIR ? t_l * u_l : n_l * v_l;
        fr_t = YDIR ? t_r * u_r : n_r * v_r;
        ft = (s_r * fl_t - s_l * fr_t + ss * (t_r - t_l)) * denom;
    } else {
        const double w_r = u_r - s_r, w_l = u_l - s_l;
        const double denom_star = h_r * w_r - h_l * w_l;
        const double num = s_l * h_r * w_r - s_r * h_l * w_l;
        const bool big = denom_star < -DRY_TOLERANCE;
        const bool left = (big & (num <= 0.0)) | (!big & (u_l + u_r >= 0.0));
        ft = f.fh * (left ? v_l : v_r);
    }
    // outside the star region the flux is that of the upwind state
    if (DRY || __builtin_expect(__any(use & !((s_l < 0.0) & (s_r > 0.0))), 0)) {
        if (HLLC) {
            fl_t = YDIR ? t_l * u_l : n_l * v_l;
            fr_t = YDIR ? t_r * u_r : n_r * v_r;
        }
        const bool left = s_l >= 0.0, right = s_r <= 0.0;
        f.fh = left ? n_l : (right ? n_r : f.fh);
        fn = left ? fl_n : (right ? fr_n : fn);
        ft = left ? fl_t : (right ? fr_t : ft);
    }
    f.fhu = YDIR ? ft : fn;
    f.fhv = YDIR ? fn : ft;
    f.a = h_r * h_r - R.h * R.h;
    f.c = h_l * h_l;
    f.d = L.h * L.h;
    return f;
}

// face_flux of the row path; `use`: the lanes whose face is used.
template <bool HLLC, bool YDIR>
__device__ __forceinline__ Face face_row(double g, const FState& L, double bL, const FState& R, double bR, bool use) {
    const double b_max = vmax(bL, bR);
    const double h_l = vmax(L.h + bL - b_max, 0.0);
    const double h_r = vmax(R.h + bR - b_max, 0.0);
    const double low = vmin(vmin(L.h, R.h), vmin(h_l, h_r));
    if (__builtin_expect(__any(use & !(low > DRY_TOLERANCE)), 0)) return face_row_as<HLLC, YDIR, true>(g, L, R, h_l, h_r, use);
    return face_row_as<HLLC, YDIR, false>(g, L, R, h_l, h_r, use);
}

// Net flux divergence of one cell from its four faces,
// rki_kernel_flux.F90:358-369 (rdx, rdy: reciprocals of dx, dy): the terms of
// the y faces, then the sum.
struct YPart {
    double fh, fhu, fhv, press;
};

enum : int { DIV_PLAIN, DIV_SHARED, DIV_TWO_OP };   // how a quotient by the spacing is taken

template <int MODE>
__device__ __forceinline__ double over(double n, const Spacing& s) {
    return MODE == DIV_PLAIN ? n / s.r.d : sdiv<MODE == DIV_TWO_OP>(n, s);
}

template <int MODE>
__device__ __forceinline__ YPart divergence_y(double g, const Spacing& dy, const Face& yb, const Face& yt) {
    YPart y;
    y.fh = over<MODE>(yt.fh - yb.fh, dy);
    y.fhu = over<MODE>(yt.fhu - yb.fhu, dy);
    y.fhv = over<MODE>(yt.fhv - yb.fhv, dy);
    y.press = over<MODE>(0.5 * g * (yb.a - yt.c + yt.d), dy);
    return y;
}

template <int MODE>
__device__ __forceinline__ void divergence(double g, const Spacing& dx, const Face& xl, const Face& xr, const YPart& y,
                                           double& fh, double& fhu, double& fhv) {
    const double half_g = 0.5 * g;
    fh = over<MODE>(-(xr.fh - xl.fh), dx) - y.fh;
    fhu = over<MODE>(-(xr.fhu - xl.fhu), dx) - y.fhu - over<MODE>(half_g * (xl.a - xr.c + xr.d), dx);
    fhv = over<MODE>(-(xr.fhv - xl.fhv), dx) - y.fhv - y.press;
}

// Clamp + KP07 desingularization + Froude backstop,
// rki_kernel_fused.F90:234-260 and :440-463.
__device__ __forceinline__ void clamp_desing(double g, double& h, double& hu, double& hv) {
    const double eps4 = 5.062499999999998e-16;  // DESING_EPS**4 folded (0x3CC23D5504170727)
    if (h < 0.0) {
        h = 0.0; hu = 0.0; hv = 0.0;
    } else if (h < DRY_TOLERANCE) {
        hu = 0.0; hv = 0.0;
    } else {
        const double h4 = pow4(h);
        if (h4 < eps4) {
            const double r = sqrt(h4 + eps4);
            const double u = SQRT2 * h * hu / r;
            const double v = SQRT2 * h * hv / r;
            hu = h * u;
            hv = h * v;
        }
        const double speed_sq = (hu * hu + hv * hv) / (h * h);
        const double fr_max_sq = (FROUDE_BACKSTOP * FROUDE_BACKSTOP * g) * h;
        if (speed_sq > fr_max_sq) {
            const double fr_scale = sqrt(fr_max_sq / speed_sq);
            hu = hu * fr_scale;
            hv = hv * fr_scale;
        }
    }
}

struct SourceTerms {
    double g;
    double n_sq;        // manning_n**2
    int has_friction;   // manning_n > 0
    int has_coriolis;   // |f| > 1e-20
    double cosf, sinf;  // cos(f dt), sin(f dt)
    double coriolis_f;  // f (used by the reverse sweep's d/d dt)
};

// Surface forcing at one cell (rki_surface_forcing.F90): wind stress (Pa),
// the central pressure gradient (Pa/m) and the precipitation rate (m/s).
struct Frc {
    double wx, wy, dpdx, dpdy, rain;
};

// Euler update + clamp + Manning + forcing + Coriolis + precipitation,
// rki_kernel_fused.F90:228-290.  With NF the Manning coefficient is the
// cell's own n_cell (friction where n_cell > 0) instead of the scalar one;
// FRC applies the surface forcing f (forcing_active).
template <bool NF, bool FRC = false>
__device__ __forceinline__ void stage_body(const SourceTerms& s, double dt, double fh, double fhu,
                                           double fhv, double& h, double& hu, double& hv, double n_cell,
                                           const Frc& f = Frc{}) {
    h = h + dt * fh;
    hu = hu + dt * fhu;
    hv = hv + dt * fhv;
    clamp_desing(s.g, h, hu, hv);
    const bool friction = NF ? (n_cell > 0.0) : (s.has_friction != 0);
    const double n_sq = NF ? n_cell * n_cell : s.n_sq;
    if (h > DRY_TOLERANCE) {
        if (friction) {
            const double u = hu / h;
            const double v = hv / h;
            const double speed = sqrt(u * u + v * v);
            const double cf = s.g * n_sq / crm::pow13(h);
            const double denom = 1.0 + dt * cf * speed / h;
            hu = hu / denom;
            hv = hv / denom;
        }
        if (FRC) {   // rki_kernel_fused.F90:273-280
            hu = hu + dt * f.wx / RHO_WATER;
            hv = hv + dt * f.wy / RHO_WATER;
            hu = hu - dt * h * f.dpdx / RHO_WATER;
            hv = hv - dt * h * f.dpdy / RHO_WATER;
        }
        if (s.has_coriolis) {
            const double hu_old = hu, hv_old = hv;
            hu = hu_old * s.cosf + hv_old * s.sinf;
            hv = -hu_old * s.sinf + hv_old * s.cosf;
        }
    }
    if (FRC) h = h + dt * f.rain;   // every cell, :286-289
}

// clamp_desing of the row path: dry cells by selects, and clamp_desing itself
// where a lane is in the KP07 band or near the Froude backstop.  The band,
// ((h h) h) h < DESING_EPS^4, is h < KP07_DEPTH: the product is monotone in h,
// also rounded.  The backstop test (hu^2 + hv^2) / h^2 > fr_max_sq is decided
// without the quotient: num < h^2 (fr_max_sq (1 - 2^-50)), rounded, implies
// num / h^2 < fr_max_sq exactly, hence the rounded quotient is at most
// fr_max_sq (a double).  Returns true where the cell update has to be redone
// with plain divisions: a lane's values are huge or not finite, or a depth is
// the dry tolerance itself.
constexpr double KP07_DEPTH = 0x1.3a92a30553261p-13;   // the smallest h with h^4, rounded, >= DESING_EPS^4

__device__ __forceinline__ bool clamp_row(double g, double& h, double& hu, double& hv) {
    const double num = hu * hu + hv * hv;
    const double fr_max_sq = (FROUDE_BACKSTOP * FROUDE_BACKSTOP * g) * h;
    const double lim = (h * h) * (fr_max_sq * (1.0 - 0x1p-50));
    const bool dry = h < DRY_TOLERANCE;
    if (__builtin_expect(__any(!(dry | ((h >= KP07_DEPTH) & (num < lim) & (h < 0x1p100)))), 0)) {
        if (__any(!((h < 0x1p100) & (num < 0x1p200)) | (h == DRY_TOLERANCE))) return true;
        clamp_desing(g, h, hu, hv);
        return false;
    }
    h = vmax(h, 0.0);
    hu = dry ? 0.0 : hu;
    hv = dry ? 0.0 : hv;
    return false;
}

// stage_body of the row path; returns true as clamp_row does.  A cell below
// the dry tolerance has zero momenta and passes through friction and
// Coriolis unchanged, the depth being raised to the tolerance for the
// quotients.  The speed only enters 1 + dt cf speed / h, so raising u^2 + v^2
// to 2^-700 leaves that sum as it is.  Friction's quotient by x^(1/3) (below
// 2^34) is a shared-reciprocal one: with a scalar n the caller takes the row
// path while g n^2 >= 2^-600, with a per-cell n this function asks for the
// same.
template <bool NF, bool FRC = false>
__device__ __forceinline__ bool stage_body_row(const SourceTerms& s, double dt, double fh, double fhu, double fhv,
                                               double& h, double& hu, double& hv, double n_cell, const Frc& f) {
    h = h + dt * fh;
    hu = hu + dt * fhu;
    hv = hv + dt * fhv;
    if (clamp_row(s.g, h, hu, hv)) return true;
    if (NF || s.has_friction) {
        const double hs = vmax(h, DRY_TOLERANCE);
        const Recip rh = recip(hs);
        const double u = rdiv<false>(hu, rh);
        const double v = rdiv<false>(hv, rh);
        const double speed = sqrt_pos(vmax(u * u + v * v, 0x1p-700));
        double gn2 = s.g * (NF ? n_cell * n_cell : s.n_sq);
        if (NF) {
            const bool friction = n_cell > 0.0;
            if (__any(friction & !(gn2 >= 0x1p-600))) return true;
            gn2 = friction ? gn2 : 0.0;
        }
        const double cf = rdiv<false>(gn2, recip(crm::pow13(hs)));
        const Recip rd = recip(1.0 + rdiv<false>(dt * cf * speed, rh));
        hu = rdiv<false>(hu, rd);
        hv = rdiv<false>(hv, rd);
    }
    if (FRC) {
        const bool wet = h > DRY_TOLERANCE;
        double qu = hu + dt * f.wx / RHO_WATER;
        double qv = hv + dt * f.wy / RHO_WATER;
        qu = qu - dt * h * f.dpdx / RHO_WATER;
        qv = qv - dt * h * f.dpdy / RHO_WATER;
        hu = wet ? qu : hu;
        hv = wet ? qv : hv;
    }
    if (s.has_coriolis) {
        const double hu_old = hu, hv_old = hv;
        hu = hu_old * s.cosf + hv_old * s.sinf;
        hv = -hu_old * s.sinf + hv_old * s.cosf;
    }
    if (FRC) {
        h = h + dt * f.rain;
        if (__any(!((h < 0x1p100) & (fabs(hu) + fabs(hv) < 0x1p100)))) return true;
    }
    return false;
}

// Largest |u| + a and |v| + a over the wet cells a lane has seen
// (rki_kernel_timestep.F90:56-69 before the division by dx and dy).
// Rounded division is monotone, so the largest of the per-cell speeds is
// the larger of the two maxima divided by dx and dy (cfl_max).
struct CflMax {
    double u, v;
};

// `same`: dx = dy, where one maximum of max(|u|, |v|) + a does.
__device__ __forceinline__ void cfl_row(double g, bool same, double h, double hu, double hv, CflMax& m) {
    const double eps4 = 5.062499999999998e-16;
    const double hs = vmax(h, DRY_TOLERANCE);
    const double wave_speed = sqrt_pos(g * hs);
    const double h4 = pow4(hs);
    const Recip rd = recip(sqrt_pos(h4 + eps4));
    const bool wet = h > DRY_TOLERANCE;
    if (same) {
        const double u_abs = rdiv<false>(vmax(fabs(hu), fabs(hv)) * SQRT2 * hs, rd);
        m.u = vmax(m.u, wet ? u_abs + wave_speed : 0.0);
    } else {
        const double u_abs = rdiv<false>(fabs(hu) * SQRT2 * hs, rd);
        const double v_abs = rdiv<false>(fabs(hv) * SQRT2 * hs, rd);
        m.u = vmax(m.u, wet ? u_abs + wave_speed : 0.0);
        m.v = vmax(m.v, wet ? v_abs + wave_speed : 0.0);
    }
}

// The same with plain divisions.
__device__ __forceinline__ void cfl_plain(double g, double h, double hu, double hv, CflMax& m) {
    const double eps4 = 5.062499999999998e-16;
    if (!(h > DRY_TOLERANCE)) return;
    const double wave_speed = sqrt(g * h);
    const double S = sqrt(pow4(h) + eps4);
    m.u = dmax(m.u, fabs(hu) * SQRT2 * h / S + wave_speed);
    m.v = dmax(m.v, fabs(hv) * SQRT2 * h / S + wave_speed);
}

__device__ __forceinline__ double cfl_max(const CflMax& m, bool same, double dx, double dy) {
    if (same) return dmax(m.u, m.v) / dx;
    return dmax(m.u / dx, m.v / dy);
}

// Per-cell CFL speed term, rki_kernel_timestep.F90:56-69; 0 for dry cells.
__device__ __forceinline__ double cfl_speed(double g, double dx, double dy, double h, double hu, double hv) {
    CflMax m{0.0, 0.0};
    cfl_plain(g, h, hu, hv, m);
    return cfl_max(m, false, dx, dy);
}

}  // namespace rk
