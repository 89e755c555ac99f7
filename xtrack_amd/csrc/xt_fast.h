/* xt_fast.h -- the compiled line code's common path.
 *
 * Compiled line code (xt_codegen.cpp) tracks a particle through *units*: one
 * element record, or a segment of cheap records.  A unit runs straight
 * through in registers on FState, without a branch, a call or a memory
 * access: what can send a particle off the common path -- an aperture, an
 * operand outside the ranges in which the short exact sequences below hold,
 * a zero whose sign a folded term could change -- only sets a flag.  A lane
 * that ends a unit with a flag set has its result thrown away and repeats
 * the unit from its start with the general element code (xt_ops.h) in one
 * out-of-line function, which also finds the element at which a particle is
 * lost.  A particle is lost once and the ranges cover every physical beam,
 * so the repeats are rare, and results are those of the general code bit
 * for bit.
 *
 * What bounds it.  With many waves (a million particles) the issue of vector
 * instructions, over 95 % of the cycles, on the thick ring 92 % of them polar
 * drifts: a polar drift takes 72 FP64 instructions and one quarter-rate
 * estimate here against 98, four and the range tests before, and the energy
 * fields come from registers.  Thick ring, 28,338 elements, 1,000,000
 * particles, one turn: 128.1 -> 92.4 ms (2.99 M vector instructions a wave
 * against 3.90 M; 3, 4 and 5 waves per SIMD 92.6, 92.8, 92.0 ms).  With one
 * wave per SIMD or fewer the chain of dependent operations: 64 particles
 * 13.4 -> 7.2 ms; thin six-cell lattice, 10,000 particles, 100 turns
 * 5.56 -> 1.00 ms, where the branches, calls and LDS reads of the general
 * code were most of the time.
 *
 * Exact quotients.  Every quotient, reciprocal and square root here is the
 * correctly rounded one.
 *
 * div1: q = RN(a y), r = a - q b, q' = RN(q + r y) with y = RN(1/b) is
 * RN(a/b) for every a, b (no over- or underflow).  With b in [1, 2) and u
 * the spacing of the quotient's binade, |y - 1/b| <= 2^-54, so
 * |q - a/b| <= u/2 + a 2^-54, at most u for a >= b and (1 + b)/2 u < 1.5 u
 * for a < b.  The error of q + r y is (a/b - q) times the relative error of
 * y.  A quotient lies at least u/(2B) from a midpoint of the grid (B: the
 * integer significand of b).  Next to a midpoint u/2 from q the error is
 * below that distance (Markstein's theorem: P. Markstein, IBM J. Res. Dev.
 * 34 (1990); J.-M. Muller et al., Handbook of Floating-Point Arithmetic,
 * 2nd ed., section 4.9); a midpoint 1.5 u from q would need a and b within a
 * few units of 2 and a remainder A 2^54 mod B of a few units, which has no
 * solution there; between them r may round, by far less than the distance.
 * Exhaustive over all pairs of significands at every precision from 4 to 11
 * bits: no exception (tests/test_fast_path.py).
 *
 * rcp_final: from any y within one unit in the last place of 1/b, r = 1 - b y
 * and RN(y + r y) is RN(1/b), except from the lower neighbour for a
 * significand b of all ones (1 - 2^-53 is pz of a particle near the axis): y
 * is therefore made 2^-55 too large before it is rounded, which leaves it
 * within one unit and above 1/b for such a b.  Exhaustive in the same test.
 */
#ifndef XT_FAST_H
#define XT_FAST_H

#include "xt_ops.h"

namespace xt {

struct FState {
    double x, px, y, py, zeta, s;
    double delta, rpp, rvv, inv_rvv;
    double ax, ay;   /* of the last magnet edge; stored late (axay) */
    /* bad: outside a range; out, outg: outside a local aperture, outside
       the global limit; axay: the unit sets ax and ay */
    bool bad, out, outg, axay;
    uint32_t ones;   /* all ones: a case that f_polar leaves out was met */
};

XT_HD uint32_t low_word(const double v) {
    uint64_t u;
    __builtin_memcpy(&u, &v, 8);
    return (uint32_t)u;
}

XT_HD bool is_neg_zero(const double v) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_class(v, 0x20);
#else
    return v == 0.0 && __builtin_signbit(v);
#endif
}

/* estimates of 1/b and 1/sqrt(x) of at least 20 correct bits */
XT_HD double est_rcp(const double b) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcp(b);
#else
    return (double)(float)(1.0 / b);
#endif
}
XT_HD double est_rsq(const double x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rsq(x);
#else
    return (double)(float)(1.0 / XT_SQRT(x));
#endif
}

/* RN(a/b) from y = RN(1/b) (above) */
XT_HD double div1(const double a, const double b, const double y) {
    const double q = a * y;
    const double r = XT_FMA(-q, b, a);
    return XT_FMA(r, y, q);
}

XT_HD double rcp_final(const double b, const double y0, const double t) {
    const double y = XT_FMA(y0, t + 0x1p-55, y0);
    const double r = XT_FMA(-b, y, 1.0);
    return XT_FMA(r, y, y);
}

/* RN(1/b) from y0 with |1 - b y0| <= 2^-28: one Newton step */
XT_HD double rcp_seeded(const double b, const double y0) {
    return rcp_final(b, y0, XT_FMA(-b, y0, 1.0));
}

/* RN(1/b): a third-order step y (1 + e + e^2) on the estimate */
XT_HD double rcp_est(const double b) {
    const double y0 = est_rcp(b);
    const double e = XT_FMA(-b, y0, 1.0);
    return rcp_final(b, y0, XT_FMA(e, e, e));
}

/* RN(sqrt(x)) by the steps of sqrt_ir (xt_ops.h), x in [2^-32, 2^32], and
   y0 = 1/sqrt(x) to 2^-30 or better */
XT_HD double sqrt_seed(const double x, double *y0) {
    const double y = est_rsq(x);
    double g = x * y;
    double h = y * 0.5;
    const double r = XT_FMA(-h, g, 0.5);
    g = XT_FMA(g, r, g);
    h = XT_FMA(h, r, h);
    double d = XT_FMA(-g, g, x);
    g = XT_FMA(d, h, g);
    d = XT_FMA(-g, g, x);
    *y0 = h + h;
    return XT_FMA(d, h, g);
}

/* ---- guards ---------------------------------------------------------------- */
/* Energy fields of the common path: |delta| <= 1/4, rvv in [1/2, 2] (with
   its reciprocal), rpp in (0, 4].  Implies the ranges of PState's fast_ok
   and polar_ok. */
XT_HD bool f_energy_ok(const double delta, const double rpp, const double rvv,
                       const double inv_rvv) {
    return delta >= -0.25 && delta <= 0.25 && rvv >= 0.5 && rvv <= 2.0 && rpp > 0.0 &&
           rpp <= 4.0 && inv_rvv >= 0.5 && inv_rvv <= 2.0;
}

/* Coordinates of at most 1: from there the generator bounds the growth
   through the following maps, so that no operand overflows. */
XT_HD void f_guard_range(FState &p) {
    p.bad |= !(xfabs(p.x) <= 1.0) | !(xfabs(p.y) <= 1.0) | !(xfabs(p.px) <= 1.0) |
             !(xfabs(p.py) <= 1.0);
}

/* px, py and zeta other than -0: the terms that a folded kick leaves out are
   zeros of either sign, and adding one changes only a sum of -0.  A sum
   with one term other than -0 is never -0, so drifts, kicks and rotations in
   a bend keep this. */
XT_HD void f_guard_signs(FState &p) {
    p.bad |= is_neg_zero(p.px) | is_neg_zero(p.py) | is_neg_zero(p.zeta);
}

/* ---- maps (the expressions of xt_ops.h) -------------------------------------- */
XT_HD void f_drift(FState &p, const double length) {
    const double xp = p.px * p.rpp;
    const double yp = p.py * p.rpp;
    const double dzeta = 1 - p.inv_rvv * (1. + (xp * xp + yp * yp) / 2.);
    p.x = p.x + xp * length;
    p.y = p.y + yp * length;
    p.s = p.s + length;
    p.zeta = p.zeta + length * dzeta;
}

/* |px|, |py| <= 1/4: the radicand lies in [0.4, 1.6] */
XT_HD void f_drift_exact(FState &p, const double length) {
    p.bad |= !(xfabs(p.px) <= 0.25) | !(xfabs(p.py) <= 0.25);
    const double px = p.px, py = p.py;
    const double one_plus_delta = 1. + p.delta;
    double y0;
    const double pz = sqrt_seed(one_plus_delta * one_plus_delta - px * px - py * py, &y0);
    const double one_over_pz = rcp_seeded(pz, y0);
    const double dzeta = 1 - p.inv_rvv * one_plus_delta * one_over_pz;
    p.x = p.x + px * one_over_pz * length;
    p.y = p.y + py * one_over_pz * length;
    p.zeta = p.zeta + dzeta * length;
    p.s = p.s + length;
}

/* Entry condition of a chain of polar drifts; the generator has bounded
   px by 1/4 and x by |rho|/2 through the chain from these (polar_plan). */
XT_HD void f_polar_guard(FState &p, const double px_max) {
    p.bad |= !(xfabs(p.x) <= 1.0) | !(xfabs(p.px) <= px_max) | !(xfabs(p.py) <= 0.25);
}

/* Polar drift (track_magnet_drift.h:45-87, polar_drift in xt_ops.h).  SMALL:
   the chain keeps |sa px / (ca pz)| <= 2^-14.5.  Then 1/(ca - sa px/pz) starts
   from ica (1 + w), w = ica sa px/pz, wrong by w^2 < 2^-28, and the quotient
   t/den by den = 1 - q4 from t + t (d + d^2 + d^3 + d^4), d = 1 - den exact: q
   is within one unit of t/den, y = 1 + (d + ...) is wrong by half a unit plus
   2^-53 d, less than the 2^-53 2 d that the final correction allows -- but
   for den = 1 - 2^-53 and t a power of two, whose correction ends in a tie
   (`ones`).
   Bound: FP64 issue.  72 instructions and one quarter-rate estimate per drift
   against 98 and four of polar_drift_ir. */
template <bool SMALL>
XT_HD void f_polar(FState &p, const double length, const double rho, const double ca,
                   const double sa, const double t2, const double ica) {
    const double x = p.x, y = p.y, px = p.px, py = p.py;
    const double one_plus_delta = p.delta + 1.0;
    const double rad = one_plus_delta * one_plus_delta - px * px - py * py;
    double y0;
    const double pz = sqrt_seed(rad, &y0);
    const double _pz = rcp_seeded(pz, y0);
    const double pxt = px * _pz;
    const double sapxt = sa * pxt;
    const double tden = ca - sapxt;
    double _ptt;
    if constexpr (SMALL)
        _ptt = rcp_seeded(tden, XT_FMA(ica, sapxt * ica, ica));
    else
        _ptt = rcp_est(tden);
    const double xr = x + rho;
    const double pst = xr * sa * _pz * _ptt;
    p.x = (x + rho * (t2 + sapxt)) * _ptt;
    p.px = ca * px + sa * pz;
    p.y = y + pst * py;
    double dz;
    if constexpr (DzReassoc<double>::value) {
        dz = length - div1(one_plus_delta * pst, p.rvv, p.inv_rvv);
    } else {
        const double t = div1(div1(one_plus_delta * xr * sa, ca, ica), pz, _pz);
        const double den = 1 - div1(div1(px * sa, ca, ica), pz, _pz);
        double q;
        if constexpr (SMALL) {
            const double d = 1.0 - den;
            double w = XT_FMA(d, d, d);
            w = XT_FMA(w, d, d);
            w = XT_FMA(w, d, d);
            q = XT_FMA(t, w, t);
            const double r = XT_FMA(-q, den, t);
            q = XT_FMA(r, 1.0 + w, q);
            const uint32_t one = low_word(den) & ~low_word(t);
            p.ones = p.ones > one ? p.ones : one;
        } else {
            q = div1(t, den, rcp_est(den));
        }
        dz = length - div1(q, p.rvv, p.inv_rvv);
    }
    p.zeta = p.zeta + dz;
    p.s = p.s + length;
}

/* kick_curvature of xt_ops.h */
XT_HD void f_curvature(FState &p, const double x, const double y, const bool has_hl,
                       const bool has_g0, const bool has_h1, const double hl, const double g0,
                       const double h1) {
    double dpx = 0.0, dpy = 0.0, dzeta = 0.0;
    bool hx = false;
    if (has_hl) {
        dpx = hl * (1. + p.delta);
        hx = true;
        dzeta = -p.inv_rvv * hl * x;
    }
    if (has_g0) {
        const double t = g0 * x;
        dpx = hx ? dpx + t : t;
        hx = true;
    }
    if (has_h1) {
        const double t = h1 * (-x * x + 0.5 * y * y);
        dpx = hx ? dpx + t : t;
        hx = true;
        dpy = h1 * x * y;
    }
    if (hx) p.px = p.px + dpx;
    if (has_h1) p.py = p.py + dpy;
    if (has_hl) p.zeta = p.zeta + dzeta;
}

/* One plane of the thick quadrupole: u, up the coordinate and slope, K the
   focusing (exact reciprocal yk), S, C its sine- and cosine-like functions;
   returns the plane's sum of the path-length terms. */
template <bool PLUS0>
XT_HD double f_quad_plane(const double u, const double up, const double K, const double yk,
                          const double S, const double C, const double length, double *u_out,
                          double *a_sum) {
    double A = -K * u;
    if (PLUS0) A = A + 0.0;   /* "- k0 + h" with zero k0, h: -0 becomes +0 */
    *u_out = u * C + up * S;
    *a_sum = A * S + up * C;
    const double AA = A * A, BB = up * up, K2 = 2.0 * K, AB = A * up;
    const double y2 = 0.5 * yk;
    return -div1(AA * C * S, K2, y2) + (BB * C * S) / 2.0 + div1(AA * length, K2, y2) +
           (BB * length) / 2.0 - div1(AB * (C * C), K, yk) + div1(AB, K, yk);
}

/* Thick quadrupole without bending (dipole_quad_map of xt_ops.h with k0 = h =
   0, where its terms in k0 and h are zeros): the generator checks that
   |k1| is in [2^-20, 2^20] and the phase sqrt(2 |k1|) length in [2^-20, pi/4].
   px and py are +0 or at least 2^-960 in magnitude, so that the slopes'
   quotients do not underflow; quotients of the path length that underflow
   are lost in the length they are added to.  An element of the collider
   ring (two halves): about 280 FP64 instructions against 1340 issue slots
   of the general map, which divides 17 times with the IEEE sequence and
   evaluates the functions for each half. */
template <bool FOCUS>
XT_HD void f_quad(FState &p, const double length, const double k1_) {
    p.bad |= ((xfabs(p.px) < 0x1p-960) & (p.px != 0.0)) | ((xfabs(p.py) < 0x1p-960) & (p.py != 0.0));
    const double D = p.delta + 1;
    const double yD = rcp_est(D);
    const double k1 = div1(k1_, D, yD);
    const double Ka = FOCUS ? k1 : -k1;
    double y0;
    const double w = sqrt_seed(Ka, &y0);
    const double yw = rcp_seeded(w, y0);
    const double ya = rcp_seeded(Ka, y0 * y0);
    const double arg = w * length;
    const double sn = xt_sin_small(arg), cs = xt_cos_small(arg);
    const double sh = xt_sinh_small(arg), ch = xt_cosh_small(arg);
    const double St = div1(sn, w, yw), Sh = div1(sh, w, yw);
    const double Sx = FOCUS ? St : Sh, Cx = FOCUS ? cs : ch;
    const double Sy = FOCUS ? Sh : St, Cy = FOCUS ? ch : cs;
    const double yx = FOCUS ? ya : -ya;
    const double xp = div1(p.px, D, yD), yp = div1(p.py, D, yD);
    double x_, y_, ax, ay;
    const double lx = f_quad_plane<true>(p.x, xp, k1, yx, Sx, Cx, length, &x_, &ax);
    const double ly = f_quad_plane<false>(p.y, yp, -k1, -yx, Sy, Cy, length, &y_, &ay);
    double length_ = length;
    length_ = length_ + 0.5 * lx;
    length_ = length_ + 0.5 * ly;
    p.x = x_;
    p.y = y_;
    p.px = ax * D;
    p.py = ay * D;
    p.zeta = p.zeta + (length - div1(length_, p.rvv, p.inv_rvv));
    p.s = p.s + length;
}

XT_HD void f_edge_linear(FState &p, const double r21, const double r43) {
    p.px = p.px + r21 * p.x;
    p.py = p.py + r43 * p.y;
}

XT_HD void f_edge_axay(FState &p, const double ca, const double cb) {
    p.ax = ca * (p.y - 0.0);
    p.ay = cb * (p.x - 0.0);
}

XT_HD void f_xy_shift(FState &p, const double ax, const double ay) {
    p.x = p.x + ax;
    p.y = p.y + ay;
}

/* op_s_shift of xt_ops.h */
XT_HD void f_s_shift(FState &p, const double ds) {
    f_drift_exact(p, ds);
    p.zeta = p.zeta + (-ds);
    p.s = p.s + (-ds);
}

XT_HD void f_s_rot(FState &p, const double sin_z, const double cos_z) {
    const double x = p.x, y = p.y, px = p.px, py = p.py;
    p.x = cos_z * x + sin_z * y;
    p.y = -sin_z * x + cos_z * y;
    p.px = cos_z * px + sin_z * py;
    p.py = -sin_z * px + cos_z * py;
}

XT_HD void f_limit_rect(FState &p, const double min_x, const double max_x, const double min_y,
                        const double max_y) {
    p.out |= !(p.x >= min_x) | !(p.x <= max_x) | !(p.y >= min_y) | !(p.y <= max_y);
}

/* min = -max in both planes: the same comparisons on the magnitudes */
XT_HD void f_limit_rect_sym(FState &p, const double max_x, const double max_y) {
    p.out |= !(xfabs(p.x) <= max_x) | !(xfabs(p.y) <= max_y);
}

XT_HD void f_limit_ellipse(FState &p, const double a_squ, const double b_squ,
                           const double a_b_squ) {
    p.out |= !(p.x * p.x * b_squ + p.y * p.y * a_squ <= a_b_squ);
}

XT_HD void f_global_aper(FState &p) {
    p.outg |= !(xfabs(p.x) <= GLOBAL_XY_LIMIT) | !(xfabs(p.y) <= GLOBAL_XY_LIMIT);
}

/* ---- the particle loop over units --------------------------------------------- */
XT_HD bool wave_any(const bool v) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ballot_w64(v) != 0;
#else
    return v;
#endif
}

/* the particle's slots (XS_*): dynamic LDS of the launch, wave-major */
XT_HD double *thread_slots(double *host_slots, int32_t *stride) {
#if defined(__HIP_DEVICE_COMPILE__)
    (void)host_slots;
    extern __shared__ double slow_lds[];
    *stride = 64;
    return slow_lds + (threadIdx.x >> 6) * (XS_N * 64) + (threadIdx.x & 63);
#else
    *stride = 1;
    return host_slots;
#endif
}

/* A unit of n elements from element e with the general element code, on the
   state in the particle's slots; with `record` (flag_monitor's value), the
   monitor or feature record of the state before it.  n = 0: the record only.
   at_element: the particle's at the unit's first element.  A lost particle is
   stored, with the element of the unit where it was lost; returns false for it.
   The number in P.state is loaded for the records alone: the elements only
   set it, and a function call would wait for the load.
   Out of line: its registers and calls take no part in the common path. */
template <bool BT, class Runner>
XT_HD_COLD bool track_unit_general(const Runner run, const typename Runner::Key key,
                                      double *host_slots, const int64_t i, const MonRef mon,
                                      const uint64_t flags, const double line_length,
                                      const int32_t e, const int32_t n, const int64_t at_turn,
                                      const int64_t at_element, const int32_t record) {
    const xtm_particles &P = *mon.P;
    const TrackCtx c{flags, line_length, P.q0, P.t_sim, 0};
    PState<double> p;
    p.slow = thread_slots(host_slots, &p.slow_stride);
    p.x = p.get(XS_X); p.px = p.get(XS_PX); p.y = p.get(XS_Y); p.py = p.get(XS_PY);
    p.zeta = p.get(XS_ZETA);
    p.chi = 1.0;
    p.at_turn = at_turn;
    p.state = record ? P.state[i] : 1;
    if (record == 3)
        feature_hook(mon.F, i, p.x, p.px, p.y, p.py, at_turn);
    else if (record)
        monitor_record(*mon.M, P, i, p.x, p.px, p.y, p.py, p.zeta, p.delta(), p.rpp(), p.rvv(),
                       p.s(), p.chi, p.at_turn, p.state, at_element, BT);
    int64_t j = 0;
    if (n > 0) {
        refresh_flags(p);
        const PRef m{&P, i};
        if (n > 1) j = run.segment(p, m, key, c, e);
        else run(p, m, key, c);
        if (c.freeze_long()) p.zeta = p.get(XS_ZETA0);
    }
    if (p.state <= 0) {
        P.x[i] = p.x; P.px[i] = p.px; P.y[i] = p.y; P.py[i] = p.py;
        P.zeta[i] = p.zeta; P.delta[i] = p.delta();
        P.rpp[i] = p.rpp(); P.rvv[i] = p.rvv(); P.s[i] = p.s();
        P.at_element[i] = BT ? at_element - j : at_element + j;
        P.at_turn[i] = at_turn; P.state[i] = p.state;
        return false;
    }
    p.put(XS_X, p.x); p.put(XS_PX, p.px); p.put(XS_Y, p.y); p.put(XS_PY, p.py);
    p.put(XS_ZETA, p.zeta);
    return true;
}

/* One particle with chi == 1 through num_ele_track elements from ele_start
   for num_turns turns (track_particle_loop of xt_ops.h with the units of the
   file comment).  BT: backtracking; the runner's elements are then the line's
   in reverse order with their backtracking programs, and ele_start counts in
   that order.  Element-by-element records (flag_monitor 2) are the host
   build's: the library takes them on the interpreter.  All lanes of a wave walk the units together; a lane without a
   particle, or whose particle is lost, takes part without effect (alive
   false), so that the loops are scalar. */
template <bool BT, class Runner>
XT_HD void track_particle_units(const xtm_particles &P, const int64_t i, bool alive,
                                const Runner &run, const TrackCtx &c, const int32_t num_turns,
                                const int32_t ele_start, const int32_t num_ele_track,
                                const int32_t flag_end_turn_actions, const int32_t flag_reset_s,
                                const int32_t flag_monitor, const MonRef &mon) {
    if (!wave_any(alive)) return;
#if defined(__HIP_DEVICE_COMPILE__)
    double *const host_slots = nullptr;
#else
    double host_slots[XS_N];
#endif
    int32_t stride;
    double *slot = thread_slots(host_slots, &stride);
    FState p = {};
    int64_t at_turn = 0, at_el = 0;   /* at_el: at_element at ele_start */
    if (alive) {
        p.x = P.x[i]; p.px = P.px[i]; p.y = P.y[i]; p.py = P.py[i];
        p.zeta = P.zeta[i]; p.s = P.s[i];
        p.delta = P.delta[i]; p.rpp = P.rpp[i]; p.rvv = P.rvv[i];
        p.inv_rvv = 1. / p.rvv;
        at_turn = P.at_turn[i];
        at_el = P.at_element[i];
        slot[XS_DELTA * stride] = p.delta;
        slot[XS_RPP * stride] = p.rpp;
        slot[XS_RVV * stride] = p.rvv;
        slot[XS_INV_RVV * stride] = p.inv_rvv;
        slot[XS_ZETA0 * stride] = p.zeta;
    }
    const int32_t ele_stop = ele_start + num_ele_track;
    bool e_ok = f_energy_ok(p.delta, p.rpp, p.rvv, p.inv_rvv);
    bool axay = false;    /* p.ax and p.ay are not stored yet */

    auto store_axay = [&]() {
        if (axay && alive) {
            mon.P->ax[i] = p.ax;
            mon.P->ay[i] = p.ay;
        }
        axay = false;
    };
    /* the general code on the unit; false when the particle is lost */
    auto general = [&](FState &q, const typename Runner::Key key, const int32_t e,
                       const int32_t n, const int32_t record) {
        slot[XS_X * stride] = p.x; slot[XS_PX * stride] = p.px;
        slot[XS_Y * stride] = p.y; slot[XS_PY * stride] = p.py;
        slot[XS_ZETA * stride] = p.zeta; slot[XS_S * stride] = p.s;
        const int64_t k = e - ele_start;
        const bool kept = track_unit_general<BT>(run, key, host_slots, i, mon, c.flags,
                                                 c.line_length, e, n, at_turn,
                                                 BT ? at_el - k : at_el + k, record);
        q.x = slot[XS_X * stride]; q.px = slot[XS_PX * stride];
        q.y = slot[XS_Y * stride]; q.py = slot[XS_PY * stride];
        q.zeta = slot[XS_ZETA * stride]; q.s = slot[XS_S * stride];
        q.delta = slot[XS_DELTA * stride]; q.rpp = slot[XS_RPP * stride];
        q.rvv = slot[XS_RVV * stride]; q.inv_rvv = slot[XS_INV_RVV * stride];
        return kept;
    };

    for (int32_t iturn = 0; iturn < num_turns; iturn++) {
        if (BT && flag_end_turn_actions > 0) {
            at_turn -= 1;
            at_el = c.num_ele_line;
            if (flag_reset_s > 0) p.s = c.line_length;
        }
        typename Runner::Key key{};
        if (ele_start < ele_stop) key = run.key(ele_start);
        if (!BT && (flag_monitor == 1 || flag_monitor == 3)) {
            store_axay();
            FState q = p;
            if (alive) general(q, key, ele_start, 0, flag_monitor);
        }
        for (int32_t e = ele_start; e < ele_stop;) {
            int32_t n = 1;
            const int32_t span = Runner::span(key);
            if (span > 1 && flag_monitor != 2 && span <= ele_stop - e) n = span;
            const typename Runner::Key next = run.key(e + n < ele_stop ? e + n : e);
            FState q = p;
            q.bad = !e_ok;
            q.out = q.outg = q.axay = false;
            q.ones = 0;
            if (flag_monitor == 2) q.bad = true;
            else if (n > 1) run.fast_segment(q, key);
            else run.fast(q, key);
            q.bad |= (q.out & !c.ignore_local()) | (q.outg & !c.ignore_global()) |
                     (q.ones == 0xffffffffu);
            if (c.freeze_long()) q.zeta = slot[XS_ZETA0 * stride];
            q.bad &= alive;
            if (__builtin_expect(wave_any(q.bad), 0)) {
                store_axay();
                if (q.bad) {
                    alive = general(q, key, e, n, flag_monitor == 2 ? 2 : 0);
                    e_ok = f_energy_ok(q.delta, q.rpp, q.rvv, q.inv_rvv);
                } else if (q.axay && alive) {
                    mon.P->ax[i] = q.ax;
                    mon.P->ay[i] = q.ay;
                }
                if (!wave_any(alive)) return;
            } else {
                axay |= q.axay;
            }
            p = q;
            e += n;
            key = next;
        }
        /* backwards also a record of flag_monitor 1, as in track_particle_loop */
        if (flag_monitor == 2 || (BT && flag_monitor == 1)) {
            store_axay();
            FState q = p;
            if (alive) general(q, key, ele_stop, 0, BT ? flag_monitor : 2);
        }
        if (!BT && flag_end_turn_actions > 0) {
            at_turn += 1;
            at_el = 0;
            if (flag_reset_s > 0) p.s = 0.;
        } else {
            at_el += BT ? -num_ele_track : num_ele_track;
        }
    }
    store_axay();
    if (alive) {
        P.x[i] = p.x; P.px[i] = p.px; P.y[i] = p.y; P.py[i] = p.py;
        P.zeta[i] = p.zeta; P.delta[i] = p.delta;
        P.rpp[i] = p.rpp; P.rvv[i] = p.rvv; P.s[i] = p.s;
        P.at_element[i] = at_el;
        P.at_turn[i] = at_turn;
    }
}

}  // namespace xt

#endif /* XT_FAST_H */
