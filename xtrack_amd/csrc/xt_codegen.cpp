// xt_codegen.cpp -- line code generation.
//
// The element-program interpreter (xt_ops.h: run_element) reads every op
// word and constant of an element from memory and dispatches on the op at
// run time.  For a line with few distinct element records (a ring is made
// of a handful of magnet, drift and aperture types repeated thousands of
// times) this file writes the same op sequence as straight-line code, with
// the constants as exact hexadecimal literals, so the device compiler sees
// constants instead of loads and no per-op dispatch remains; the per-element
// dispatch becomes one switch on a 32-bit record index.  Folded
// multipole-kick passes are unrolled with the zero pattern of their
// coefficients known.
//
// There are two codes of a record.  Its general code (Gen) calls the element
// functions that the interpreter calls, with the values the interpreter would
// load.  Its unit code (FastGen) runs the maps of xt_fast.h on the state in
// registers, under guards; a particle that fails one repeats the unit in the
// general code.  Both give the interpreter's bits.  A line whose elements
// mostly have no unit code has general code alone.
#include <cinttypes>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <algorithm>
#include <cstring>
#include <map>
#include <tuple>
#include <string>
#include <vector>

#include "../../include/xtrack_amd.h"
#include "xt_codegen.h"
#include "xt_program.h"

namespace {

int64_t wbits(double d) { int64_t u; std::memcpy(&u, &d, 8); return u; }

// exact literal for a double
std::string lit(double v) {
    if (std::isnan(v)) return "__builtin_nan(\"\")";
    if (std::isinf(v)) return v > 0 ? "__builtin_inf()" : "(-__builtin_inf())";
    char buf[64];
    std::snprintf(buf, sizeof buf, "%a", v);
    std::string s(buf);
    if (s[0] == '-') return "(" + s + ")";
    return s;
}

const int kNargs[OP_NUM] = XT_OP_NARGS_INIT;

// Records whose arithmetic is at most this many ops (a kick pass counts
// its terms) and that hold no integrator, map or RF op are cheap enough
// for the per-element dispatch to matter; runs of them form segments.
constexpr int kSmallCost = 12;
constexpr size_t kSegMax = 31;           // elements per segment (< 32)
constexpr int64_t kSegMaxCount = 256;    // distinct segments per line
constexpr int64_t kSegMaxBody = 2048;    // sum of their lengths
constexpr int64_t kSegOnceBody = 512;    // the same with segments used once
// line code: every record literal up to this many distinct records, else
// literal only for records used more than once whose structure occurs with
// at most kLiteralPerStruct constant sets, at most kLiteralMax of them
constexpr int64_t kLiteralAll = 64;
constexpr int64_t kLiteralMax = 1024;
constexpr int64_t kLiteralPerStruct = 4;
static_assert(kSegMax <= XT_KEY_SPAN_MASK, "segment length must fit its key field");

struct Gen {
    const std::vector<double> &prog;
    const int64_t base;   // program offset of the record
    const bool loads;     // constants as loads rp[k] instead of literals
    const bool rel;       // program addresses relative to rp = prog + base
    std::string out;
    std::string err;
    int cost = 0;         // rough size of the record's arithmetic (ops, kick terms)
    bool heavy = false;   // holds an integrator, a map or an RF op

    Gen(const std::vector<double> &p, int64_t b, bool l, bool r = false)
        : prog(p), base(b), loads(l), rel(l || r) {}

    // constant at absolute program index i
    std::string c(int64_t i) const {
        if (loads) return "rp[" + std::to_string(i - base) + "]";
        return lit(prog[i]);
    }
    // address of program word i: relative to the record (rp) in loads mode
    // and in relative literal mode, so that records of the same structure
    // (or the same constants) in different places produce the same text
    std::string addr(int64_t i) const {
        if (rel) return "rp + " + std::to_string(i - base);
        return "prog + " + std::to_string(i);
    }
    std::string cs(int64_t i, int n) const {
        std::string s;
        for (int k = 0; k < n; k++) s += ", " + c(i + k);
        return s;
    }

    void line(const std::string &s) { out += "    " + s + "\n"; }

    bool in_range(int64_t pos, int64_t n) const {
        return pos >= 0 && n >= 0 && pos + n <= (int64_t)prog.size();
    }

    // one folded Horner pass from the coefficient block at `fp`
    bool kick_pass(int64_t fp, const std::string &w) {
        if (!in_range(fp, 1)) return false;
        const int64_t top = wbits(prog[fp]);
        if (top < 0 || !in_range(fp, 2 * top + 3)) return false;
        const int64_t ia = fp + 1, ib = fp + 2 + top;
        line("    {");
        line("        double dpx = " + c(ia + top) + ", dpy = " + c(ib + top) + ";");
        for (int64_t k = top - 1; k >= 0; k--) {
            line("        xt::horner_step(dpx, dpy, x, y, " + c(ia + k) + ", " + c(ib + k) + ", " +
                 (prog[ia + k] != 0.0 ? "true" : "false") + ", " +
                 (prog[ib + k] != 0.0 ? "true" : "false") + ");");
        }
        line("        xt::kick_pass_apply(p, " + w + ", dpx, dpy);");
        line("    }");
        cost += (int)top + 1;
        return true;
    }

    bool kick(int64_t pc) {
        const double *a = &prog[pc + 1];
        const std::string w = c(pc + 1);
        const int64_t desc = wbits(a[1]);
        const int64_t mask = wbits(a[2]);
        if (!in_range(desc, KD_ARR)) return false;
        line("if (!xt::kick_sane(p)) {");
        line("    xt::kick_literal_apply(p, " + w + ", (const double *)(" + addr(desc) + "));");
        line("} else {");
        line("    const double x = p.x, y = p.y;");
        for (int k = 0; k < 3; k++) {
            if (!(mask & (1 << k))) continue;
            if (!kick_pass(wbits(prog[desc + KD_FASTOFF + k]), w)) return false;
        }
        if (mask & (8 | 16 | 32)) {
            line(std::string("    xt::kick_curvature(p, x, y, ") + ((mask & 8) ? "true" : "false") +
                 ", " + ((mask & 16) ? "true" : "false") + ", " + ((mask & 32) ? "true" : "false") +
                 cs(pc + 4, 3) + ");");
        }
        line("}");
        return true;
    }

    bool record(int64_t pc) {
        for (int guard = 0; guard < 100000; guard++) {
            if (!in_range(pc, 1)) return false;
            const int64_t op = wbits(prog[pc]);
            if (op < 0 || op >= OP_NUM) return false;
            if (op == OP_END) return true;
            const int n = kNargs[op];
            if (!in_range(pc + 1, n)) return false;
            const int64_t a = pc + 1;
            const std::string at = addr(pc + 1);
            cost += 1;
            if (op == OP_POLAR || op == OP_DIPQUAD || op == OP_YOSHIDA4_BEND ||
                op == OP_BEND_CURVED || op == OP_BEND_STRAIGHT ||
                op == OP_YOSHIDA6_BEND || op == OP_RF_KICK || op == OP_X_ROT || op == OP_Y_ROT ||
                op == OP_RF_MULT)
                heavy = true;
            switch (op) {
            case OP_DRIFT_EXP: line("xt::drift_expanded(p" + cs(a, 1) + ");"); break;
            case OP_DRIFT_EXACT: line("xt::drift_exact(p" + cs(a, 1) + ");"); break;
            case OP_POLAR: line("xt::polar_drift(p" + cs(a, 6) + ");"); break;
            case OP_BEND_CURVED: line("xt::op_bend_curved(p" + cs(a, 9) + ");"); break;
            case OP_BEND_STRAIGHT: line("xt::op_bend_straight(p" + cs(a, 2) + ");"); break;
            case OP_DIPQUAD: line("xt::dipole_quad(p" + cs(a, 4) + ");"); break;
            case OP_YOSHIDA4_BEND: line("xt::op_yoshida4(p" + cs(a, 14) + ");"); break;
            case OP_YOSHIDA6_BEND: line("xt::op_yoshida6(p, " + at + ");"); break;
            case OP_KICK:
                if (!kick(pc)) return false;
                break;
            case OP_EDGE_AXAY: line("xt::op_edge_axay(p, m" + cs(a, 2) + ");"); break;
            case OP_EDGE_CLEAR_AXAY: line("xt::op_edge_clear_axay(m);"); break;
            case OP_EDGE_LINEAR: line("xt::op_edge_linear(p" + cs(a, 2) + ");"); break;
            case OP_RF_KICK:
                line("xt::op_rf_kick(p, m" + cs(a, 5) + ", xt::wbits(" + c(a + 5) +
                     "), c.line_length, c.q0, c.t_sim, c.kill_energy());");
                break;
            case OP_LIMIT_RECT:
                line("xt::op_limit_rect(p" + cs(a, 4) + ", c.ignore_local());");
                break;
            case OP_LIMIT_ELLIPSE:
                line("xt::op_limit_ellipse(p" + cs(a, 3) + ", c.ignore_local());");
                break;
            case OP_GLOBAL_APER: line("xt::op_global_aper(p, c.ignore_global());"); break;
            case OP_XY_SHIFT: line("xt::op_xy_shift(p" + cs(a, 2) + ");"); break;
            case OP_S_SHIFT: line("xt::op_s_shift(p" + cs(a, 1) + ");"); break;
            case OP_X_ROT: line("xt::op_x_rot(p, m" + cs(a, 3) + ");"); break;
            case OP_Y_ROT: line("xt::op_y_rot(p, m" + cs(a, 3) + ");"); break;
            case OP_S_ROT: line("xt::op_s_rot(p" + cs(a, 2) + ");"); break;
            case OP_RF_MULT:
                // the descriptor holds program offsets: absolute addressing
                line("xt::op_rf_mult(p, m, xt::cptr(prog) + " + std::to_string(pc + 1) +
                     ", xt::cptr(prog), c.q0, c.kill_energy());");
                break;
            default: return false;
            }
            pc += 1 + n;
        }
        return false;
    }
};


/* The unit code of one record or of a segment of records: the maps of
   xt_fast.h in order, with the guards that their folded forms need.  The
   generator follows bounds on |x|, |y|, |px| and |py| through the unit
   (constants known; kInf where they are loaded) and whether px, py and zeta
   can be -0, and writes a guard only where one is not already implied. */
struct FastGen {
    const std::vector<double> &prog;
    const bool loads;
    std::string out;
    bool direct = false;   // holds an op that only the general code has
    bool axay = false;     // sets ax and ay
    int gain = 0;          // of the unit over the general code in the loop (weight())

    // loaded constants that every record of the structure shares: literals
    const std::vector<char> *shared;

    FastGen(const std::vector<double> &p, bool l, const std::vector<char> *s = nullptr)
        : prog(p), loads(l), shared(s) {}

    static constexpr double kInf = 1e300;
    static constexpr double kRange = 0x1p100;   // products of a few stay finite
    static constexpr int kMaxDrifts = 64;
    int64_t base = 0;
    double bx = kInf, by = kInf, bpx = kInf, bpy = kInf;
    bool signs = false;

    std::string c(int64_t i) const {
        if (loads && !(shared && i - base < (int64_t)shared->size() && (*shared)[i - base]))
            return "rp[" + std::to_string(i - base) + "]";
        return lit(prog[i]);
    }
    std::string cs(int64_t i, int n) const {
        std::string s;
        for (int k = 0; k < n; k++) s += ", " + c(i + k);
        return s;
    }
    void line(const std::string &s) { out += "    " + s + "\n"; }

    void guard_range() {
        if (bx <= kRange && by <= kRange && bpx <= kRange && bpy <= kRange) return;
        line("xt::f_guard_range(p);");
        bx = by = bpx = bpy = 1.0;
    }
    void guard_signs() {
        if (!signs) line("xt::f_guard_signs(p);");
        signs = true;
    }

    /* Checks of one convex limit (a LimitRect, the global limit) along
       drifts: with px and py unchanged and lengths of one sign, x and y run
       monotonically (rounding is monotone), so a check between two others of
       the same limit is implied by them.  `held` is the place of the last
       check, not written yet. */
    struct Convex {
        std::string text;      // the anchored check; empty: none
        int64_t held = -1;     // place in out of the check held back
        int sign = 0;          // sign of the drift lengths since the anchor
    };
    Convex rect, glob;

    void flush(Convex &v, Convex &other) {
        if (v.held >= 0) {
            const std::string t = "    " + v.text + "\n";
            out.insert((size_t)v.held, t);
            if (other.held > v.held) other.held += (int64_t)t.size();
        }
        v = Convex();
    }
    void flush_limits() {
        flush(rect, glob);
        flush(glob, rect);
    }
    void drifted(double length) {
        const int sg = length > 0 ? 1 : length < 0 ? -1 : 0;
        for (Convex *v : {&rect, &glob}) {
            if (v->text.empty()) continue;
            if (loads || sg == 0 || (v->sign != 0 && v->sign != sg)) {
                flush(*v, v == &rect ? glob : rect);
            } else {
                v->sign = sg;
            }
        }
    }
    void convex(Convex &v, const std::string &check) {
        if (v.text == check) {
            v.held = (int64_t)out.size();
            return;
        }
        flush(v, &v == &rect ? glob : rect);
        line(check);
        v.text = check;
    }

    bool in_range(int64_t pos, int64_t n) const {
        return pos >= 0 && n >= 0 && pos + n <= (int64_t)prog.size();
    }

    struct Polar { int64_t length, consts; };   // program indices: length; ca sa t2 ica

    /* Bounds through a chain of polar drifts of curvature radius rho with
       kicks px -= kick[j] after drift j, from |x| <= 1, |px| <= p0, |py| <=
       1/4, |delta| <= 1/4: 0 when they leave the ranges of f_polar, 2 when
       its small-angle form holds, else 1; the bounds on x and px at the end. */
    int polar_plan(const std::vector<Polar> &d, const std::vector<double> &kick, double rho,
                   double p0, double *x_end, double *px_end) const {
        double xb = 1.0, lo = -p0, hi = p0;
        bool small = true;
        for (size_t j = 0; j < d.size(); j++) {
            const double ca = prog[d[j].consts], sa = prog[d[j].consts + 1];
            const double t2 = prog[d[j].consts + 2], ica = prog[d[j].consts + 3];
            if (ica == 0.0) return 0;
            const double pm = std::max(-lo, hi);
            if (!(pm <= 0.25)) return 0;
            const double pz_lo = std::sqrt(0.5625 - 0.0625 - pm * pm), pz_hi = 1.25;
            const double w = std::fabs(sa) * pm / pz_lo;
            if (!(w / ca <= 0x1.6p-15)) small = false;   // below 2^-14.5
            xb = (xb + std::fabs(rho) * (t2 + w)) / (ca - w);
            if (!(xb <= 0x1p20) || !(std::fabs(rho) >= 2 * xb)) return 0;
            const double s_lo = std::min(sa * pz_lo, sa * pz_hi);
            const double s_hi = std::max(sa * pz_lo, sa * pz_hi);
            lo = (lo < 0 ? lo : ca * lo) + s_lo;
            hi = (hi > 0 ? hi : ca * hi) + s_hi;
            if (j < kick.size()) {
                lo -= kick[j];
                hi -= kick[j];
            }
            lo -= 0x1p-40;
            hi += 0x1p-40;
        }
        if (!(std::max(-lo, hi) <= 0.25)) return 0;
        *x_end = xb;
        *px_end = std::max(-lo, hi);
        return small ? 2 : 1;
    }

    /* drifts d with kicks (program index of the strength, times the word at
       L) between them */
    void polar_chain(int64_t rho, const std::vector<Polar> &d, const std::vector<int64_t> &kick,
                     int64_t L) {
        std::vector<double> kv;
        for (int64_t k : kick) kv.push_back(prog[k] * prog[L]);
        double xe = 0, pe = 0, p0 = 0x1p-7;
        int plan = polar_plan(d, kv, prog[rho], p0, &xe, &pe);
        if (plan != 2) {
            p0 = 0x1p-4;
            plan = polar_plan(d, kv, prog[rho], p0, &xe, &pe);
        }
        if (plan == 0) {
            direct = true;
            return;
        }
        line("xt::f_polar_guard(p, " + lit(p0) + ");");
        for (size_t j = 0; j < d.size(); j++) {
            line(std::string("xt::f_polar<") + (plan == 2 ? "true" : "false") + ">(p, " +
                 c(d[j].length) + ", " + c(rho) + cs(d[j].consts, 4) + ");");
            if (j < kick.size()) line("p.px = p.px - " + c(kick[j]) + " * " + c(L) + ";");
        }
        double ell = 0;
        for (auto &v : d) ell += std::fabs(prog[v.length]);
        bx = xe;
        bpx = pe;
        bpy = 0.25;
        by += 4 * ell;
    }

    /* one folded Horner pass (xt_ops.h: horner_step, kick_pass_apply); a sum
       that is known to be zero is left out */
    bool kick_pass(int64_t fp, const std::string &w, double wv, double *dpx_b, double *dpy_b) {
        if (!in_range(fp, 1)) return false;
        const int64_t top = wbits(prog[fp]);
        if (top < -1 || top > 1000 || !in_range(fp, 2 * top + 3)) return false;
        if (top < 0) return true;
        const int64_t ia = fp + 1, ib = fp + 2 + top;
        bool zx = prog[ia + top] == 0.0, zy = prog[ib + top] == 0.0;
        line("{");
        line("    double dpx = " + (zx ? std::string("0.0") : c(ia + top)) + ", dpy = " +
             (zy ? std::string("0.0") : c(ib + top)) + ", zre, zim;");
        double b = std::fabs(prog[ia + top]) + std::fabs(prog[ib + top]);
        for (int64_t k = top - 1; k >= 0; k--) {
            if (zx && zy) return false;   // top is the highest non-zero coefficient
            line(std::string("    zre = ") + (zx ? "-(dpy * y)" : zy ? "dpx * x"
                                                                     : "dpx * x - dpy * y") + ";");
            line(std::string("    zim = ") + (zx ? "dpy * x" : zy ? "dpx * y"
                                                                  : "dpx * y + dpy * x") + ";");
            zx = zy = false;
            line("    dpx = " + (prog[ia + k] != 0.0 ? c(ia + k) + " + zre" : "zre") + ";");
            line("    dpy = " + (prog[ib + k] != 0.0 ? c(ib + k) + " + zim" : "zim") + ";");
            b = b * (bx + by) + std::fabs(prog[ia + k]) + std::fabs(prog[ib + k]);
        }
        if (!zx) line("    p.px = p.px + " + w + " * (-dpx);");
        if (!zy) line("    p.py = p.py + " + w + " * dpy;");
        line("}");
        *dpx_b += std::fabs(wv) * b;
        *dpy_b += std::fabs(wv) * b;
        return true;
    }

    bool kick(int64_t pc) {
        const double *a = &prog[pc + 1];
        const std::string w = c(pc + 1);
        const int64_t desc = wbits(a[1]), mask = wbits(a[2]);
        if (!in_range(desc, KD_ARR)) return false;
        guard_range();
        guard_signs();
        double dx = 0, dy = 0;
        line("{");
        line("const double x = p.x, y = p.y;");
        line("(void)x; (void)y;");
        for (int k = 0; k < 3; k++)
            if ((mask & (1 << k)) &&
                !kick_pass(wbits(prog[desc + KD_FASTOFF + k]), w, a[0], &dx, &dy))
                return false;
        if (mask & (8 | 16 | 32))
            line(std::string("xt::f_curvature(p, x, y, ") + ((mask & 8) ? "true" : "false") +
                 ", " + ((mask & 16) ? "true" : "false") + ", " + ((mask & 32) ? "true" : "false") +
                 cs(pc + 4, 3) + ");");
        line("}");
        dx += 2 * std::fabs(a[3]) + std::fabs(a[4]) * bx + std::fabs(a[5]) * (bx * bx + by * by);
        dy += std::fabs(a[5]) * bx * by;
        // the same code serves records with other strengths
        bpx = loads ? kInf : bpx + dx;
        bpy = loads ? kInf : bpy + dy;
        return true;
    }

    void quad(int64_t a) {
        const double L = prog[a], k0 = prog[a + 1], k1 = prog[a + 2], h = prog[a + 3];
        const double k = std::fabs(k1), ph = 4.0 / 3.0 * k * L * L;
        // phase sqrt(k1 / (1 + delta)) L in [2^-20, pi/4], |delta| <= 1/4
        if (wbits(k0) != 0 || wbits(h) != 0 || !(k >= 0x1p-20 && k <= 0x1p20) ||
            !(0.8 * k * L * L >= 0x1p-40) || !(ph <= 0.61) || !(std::fabs(L) <= 0x1p20)) {
            direct = true;
            return;
        }
        guard_range();
        guard_signs();
        gain += 200;
        line(std::string("xt::f_quad<") + (k1 > 0 ? "true" : "false") + ">(p, " + c(a) + ", " +
             c(a + 2) + ");");
        const double x = 2 * bx + 4 * std::fabs(L) * bpx, y = 2 * by + 4 * std::fabs(L) * bpy;
        bpx = 4 * bpx + 4 * k * std::fabs(L) * bx;
        bpy = 4 * bpy + 4 * k * std::fabs(L) * by;
        bx = x;
        by = y;
        if (loads) bx = by = bpx = bpy = kInf;
    }

    /* What the record gains in the loop over units against the loop over
       general code (build_code_set: units), in units of a tenth of what a
       drift, a thin kick or an aperture gains in a segment (0.1 us on 64
       particles, 0.25 us on 300,000).  Measured per element: a thick
       quadrupole 2 us, a polar drift 0.2 us, single thin elements half of
       those in segments; a record without unit code loses 0.7 to 2.4 us to its
       out-of-line call, less the more of its time is in functions that are out
       of line anyway; exact bend maps gain 0.7 us there. */
    int weight(bool small) const {
        if (direct) return gain;
        return (small ? 10 : 5) + gain;
    }

    static int drifts(int64_t op) {
        return op == OP_YOSHIDA4_BEND ? 4 : op == OP_YOSHIDA6_BEND ? 8 : op == OP_POLAR ? 1 : 0;
    }

    bool same_op(int64_t p, int64_t q) const {
        const int64_t op = wbits(prog[p]);
        return op == wbits(prog[q]) &&
               std::memcmp(&prog[p + 1], &prog[q + 1], sizeof(double) * kNargs[op]) == 0;
    }

    /* append record pc; false for a program this generator cannot read.  A
       strong bend is integrated in hundreds of equal steps: the largest
       repetition of its ops becomes a loop, and a bend that still holds more
       than kMaxDrifts polar drifts is left to the general code (straight-line
       code for 576 drifts compiles in minutes). */
    bool record(int64_t pc) {
        base = pc;
        std::vector<int64_t> ops;
        int n_drifts = 0;
        bool exact_bend = false;
        for (;;) {
            if (!in_range(pc, 1) || ops.size() > 100000) return false;
            const int64_t op = wbits(prog[pc]);
            if (op < 0 || op >= OP_NUM) return false;
            if (op == OP_END) break;
            if (!in_range(pc + 1, kNargs[op])) return false;
            ops.push_back(pc);
            n_drifts += drifts(op);
            exact_bend |= op == OP_BEND_CURVED || op == OP_BEND_STRAIGHT;
            pc += 1 + kNargs[op];
        }
        const int all_drifts = n_drifts;
        // ops [first, first + period * count) repeat the first period
        size_t first = 0, period = 0, count = 0;
        if (n_drifts > kMaxDrifts) {
            for (size_t f = 0; f < ops.size() && f < 8; f++)
                for (size_t q = 1; 2 * q <= ops.size() - f && q <= 64; q++) {
                    size_t e = f + q;
                    while (e < ops.size() && same_op(ops[e], ops[e - q])) e++;
                    const size_t r = (e - f) / q;
                    if (r > 1 && (r - 1) * q > (count ? (count - 1) * period : 0)) {
                        first = f;
                        period = q;
                        count = r;
                    }
                }
            for (size_t k = first; count && k < first + period * (count - 1); k++)
                n_drifts -= drifts(wbits(prog[ops[k]]));
            if (n_drifts > kMaxDrifts) direct = true;
        }
        // the rest of the record may still find that it is direct
        auto finish = [&]() {
            gain += direct ? (exact_bend ? 50 : -200 - 10 * all_drifts) : 20 * all_drifts;
            return true;
        };
        if (direct) return finish();
        for (size_t k = 0; k < ops.size(); k++) {
            if (count && k == first) {
                flush_limits();
                bx = by = bpx = bpy = kInf;   // as every repetition finds them
                signs = false;
                out += "#pragma clang loop unroll(disable)\n";
                line("for (int step = 0; step < " + std::to_string(count) + "; step++) {");
            }
            if (!emit(ops[k])) return false;
            if (direct) return finish();
            if (count && k == first + period - 1) {
                flush_limits();
                line("}");
                k = first + period * count - 1;
            }
        }
        return finish();
    }

    bool emit(int64_t pc) {
        const int64_t op = wbits(prog[pc]);
        const int64_t a = pc + 1;
        if (op != OP_DRIFT_EXP && op != OP_LIMIT_RECT && op != OP_LIMIT_ELLIPSE &&
            op != OP_GLOBAL_APER)
            flush_limits();
        switch (op) {
        case OP_DRIFT_EXP: {
            drifted(prog[a]);
            line("xt::f_drift(p, " + c(a) + ");");
            const double l = loads ? kInf : 8 * std::fabs(prog[a]);
            bx += l * bpx;
            by += l * bpy;
            break; }
        case OP_DRIFT_EXACT: {
            line("xt::f_drift_exact(p, " + c(a) + ");");
            const double l = loads ? kInf : 2 * std::fabs(prog[a]);
            bpx = bpy = 0.25;
            bx += l;
            by += l;
            break; }
        case OP_POLAR:
            polar_chain(a + 1, {{a, a + 2}}, {}, a);
            break;
        case OP_YOSHIDA4_BEND:
            polar_chain(a + 1, {{a + 4, a + 5}, {a + 9, a + 10}, {a + 9, a + 10},
                                {a + 4, a + 5}}, {a + 2, a + 3, a + 2}, a);
            break;
        case OP_YOSHIDA6_BEND: {
            std::vector<Polar> d;
            std::vector<int64_t> k;
            for (int j = 0; j < 8; j++) {
                const int64_t q = a + 6 + 5 * (j < 4 ? j : 7 - j);
                d.push_back({q, q + 1});
                if (j < 7) k.push_back(a + 2 + (j < 4 ? j : 6 - j));
            }
            polar_chain(a + 1, d, k, a);
            break; }
        case OP_DIPQUAD: quad(a); break;
        case OP_KICK:
            if (!kick(pc)) return false;
            break;
        case OP_EDGE_AXAY:
            line("xt::f_edge_axay(p" + cs(a, 2) + ");");
            axay = true;
            break;
        case OP_EDGE_CLEAR_AXAY:
            line("p.ax = p.ay = 0.;");
            axay = true;
            break;
        case OP_EDGE_LINEAR:
            if (!loads && prog[a] == 0.0 && prog[a + 1] == 0.0) {
                guard_range();
                guard_signs();
                break;
            }
            line("xt::f_edge_linear(p" + cs(a, 2) + ");");
            bpx = loads ? kInf : bpx + std::fabs(prog[a]) * bx;
            bpy = loads ? kInf : bpy + std::fabs(prog[a + 1]) * by;
            break;
        case OP_XY_SHIFT:
            line("xt::f_xy_shift(p" + cs(a, 2) + ");");
            bx += loads ? kInf : std::fabs(prog[a]);
            by += loads ? kInf : std::fabs(prog[a + 1]);
            break;
        case OP_S_ROT: {
            line("xt::f_s_rot(p" + cs(a, 2) + ");");
            signs = false;
            bx = by = 2 * (bx + by);
            bpx = bpy = 2 * (bpx + bpy);
            break; }
        case OP_LIMIT_RECT:
            if (!loads && prog[a] == -prog[a + 1] && prog[a + 2] == -prog[a + 3])
                convex(rect, "xt::f_limit_rect_sym(p, " + c(a + 1) + ", " + c(a + 3) + ");");
            else if (!loads)
                convex(rect, "xt::f_limit_rect(p" + cs(a, 4) + ");");
            else
                line("xt::f_limit_rect(p" + cs(a, 4) + ");");
            break;
        case OP_LIMIT_ELLIPSE:
            line("xt::f_limit_ellipse(p" + cs(a, 3) + ");");
            break;
        case OP_GLOBAL_APER: convex(glob, "xt::f_global_aper(p);"); break;
        case OP_S_SHIFT:
            line("xt::f_s_shift(p, " + c(a) + ");");
            bpx = bpy = 0.25;
            bx += loads ? kInf : 2 * std::fabs(prog[a]);
            by += loads ? kInf : 2 * std::fabs(prog[a]);
            break;
        default:
            // RF, frame rotations, exact bends: the general code
            direct = true;
            break;
        }
        return true;
    }

    std::string body() {
        flush_limits();
        if (direct) return "    p.bad = true;\n";
        if (axay) line("p.axay = true;");
        return out;
    }
};

/* Functions of the generated code for a set of lines (one line, or the
   lines of a batch).  A record whose literal code serves at least two
   elements of the set (every record, for a single line of at most
   kLiteralAll distinct records) gets a literal function; a record that
   serves one element only -- a magnet with its own field errors -- gets the
   function of its structure, shared with every record of that structure,
   which reads its constants from the program (scalar loads at
   rp = prog + entry[e]).  Literal functions for thousands of single-use
   records would be megabytes of instructions, streamed through the
   instruction cache once per turn. */
struct CodeSet {
    std::vector<std::string> body;             // function bodies (general code)
    std::vector<std::string> fast;             // their unit code
    std::vector<char> small;                   // cheap literal records
    bool units = true;                         // the loop over units (xt_fast.h)
    bool keyed_pc = false;                     // keys carry the program offset
    std::vector<std::vector<int32_t>> segs;    // segment function bodies
    std::vector<std::string> fast_segs;        // their unit code
};

// key of a function: its general and its unit code
std::string both(const std::string &general, const std::string &unit) {
    return general + '\n' + unit;
}

// the words of a record that its text loads (rp[k])
std::vector<int64_t> loaded_words(const std::string &text) {
    std::vector<int64_t> out;
    for (size_t q = text.find("rp["); q != std::string::npos; q = text.find("rp[", q + 3))
        out.push_back(std::strtoll(text.c_str() + q + 3, nullptr, 10));
    return out;
}

/* with_units: general and unit code of every function; else general code
   alone, for the element loop. */
int build_code_set(const std::vector<const std::vector<int64_t> *> &entries,
                   const std::vector<const std::vector<double> *> &progs, bool keyed_pc,
                   bool with_units, CodeSet &cs, std::vector<std::vector<int32_t>> &recs,
                   std::string &err) {
    const size_t nl = entries.size();
    cs = CodeSet();
    // a program that the unit generator does not read has no unit code
    auto unit = [&](FastGen &f, int64_t pc) {
        if (with_units && !f.record(pc)) {
            f.direct = true;
            f.gain = -200;
        }
        return with_units ? f.body() : std::string();
    };
    // distinct records of each line and their element counts
    std::vector<std::map<int64_t, int64_t>> uses(nl);
    int64_t n_distinct = 0;
    for (size_t l = 0; l < nl; l++) {
        for (int64_t e : *entries[l]) uses[l][e]++;
        n_distinct += (int64_t)uses[l].size();
    }
    const bool all_literal = !keyed_pc && nl == 1 && n_distinct <= kLiteralAll;
    cs.keyed_pc = !all_literal;
    // Structures: the general and the unit code of a record with its constants
    // as loads.  Records of one op sequence differ in the latter where a form
    // depends on the ranges of their constants.
    struct Structure {
        std::string general, unit;
        std::vector<int64_t> words;     // the program words that the texts load
        bool small = false;
        int weight = 0;
    };
    std::vector<Structure> structs;
    std::map<std::string, int32_t> struct_of;               // by both texts
    // Literals: the records of one structure with the same constants.  A record
    // is known by its structure and the words loaded there, so that literal
    // text is written only for the records that get a function of their own;
    // a line of literal records only knows them by their text, with program
    // addresses that are not relative to the record.
    struct Literal {
        size_t line;
        int64_t pc, uses;
        int32_t structure;
        std::string general, unit;
    };
    std::map<std::string, Literal> lits;
    std::vector<std::map<int64_t, std::pair<int32_t, const std::string *>>> record(nl);
    // distinct literals of a structure; heavy records of one general code count
    // together, since their units are many copies of long code otherwise
    std::map<std::string, int64_t> lits_of_struct;
    auto counted = [&](const Structure &v) {
        return v.small ? both(v.general, v.unit) : v.general;
    };
    int64_t gain = 0;
    auto cannot = [&](size_t l, int64_t pc) {
        err = "cannot generate code for line " + std::to_string(l) + " at program offset " +
              std::to_string(pc);
        return XTM_ERR_ARG;
    };
    auto write = [&](Literal &v) {
        Gen g(*progs[v.line], v.pc, false, !all_literal);
        FastGen f(*progs[v.line], false);
        const bool ok = g.record(v.pc);
        v.unit = unit(f, v.pc);
        v.general = std::move(g.out);
        return ok;
    };
    for (size_t l = 0; l < nl; l++)
        for (auto &pu : uses[l]) {
            Gen gs(*progs[l], pu.first, true);
            FastGen fs(*progs[l], true);
            if (!gs.record(pu.first)) return cannot(l, pu.first);
            const std::string fast = unit(fs, pu.first);
            const auto st = struct_of.emplace(both(gs.out, fast), (int32_t)structs.size());
            if (st.second) {
                structs.emplace_back();
                Structure &v = structs.back();
                v.small = !gs.heavy && gs.cost <= kSmallCost;
                v.weight = fs.weight(v.small);
                v.words = loaded_words(gs.out);
                for (int64_t k : loaded_words(fast)) v.words.push_back(k);
                std::sort(v.words.begin(), v.words.end());
                v.words.erase(std::unique(v.words.begin(), v.words.end()), v.words.end());
                v.general = gs.out;
                v.unit = fast;
            }
            const Structure &sv = structs[st.first->second];
            Literal lit{l, pu.first, 0, st.first->second, {}, {}};
            std::string key;
            if (all_literal) {
                if (!write(lit)) return cannot(l, pu.first);
                key = both(lit.general, lit.unit);
            } else {
                key.assign(reinterpret_cast<const char *>(&lit.structure), sizeof lit.structure);
                for (int64_t k : sv.words) {
                    if (pu.first + k < 0 || pu.first + k >= (int64_t)progs[l]->size())
                        return cannot(l, pu.first);
                    key.append(reinterpret_cast<const char *>(&(*progs[l])[pu.first + k]),
                               sizeof(double));
                }
            }
            auto ins = lits.emplace(std::move(key), std::move(lit));
            if (ins.second) lits_of_struct[counted(sv)]++;
            ins.first->second.uses += pu.second;
            gain += (int64_t)sv.weight * pu.second;
            record[l][pu.first] = {st.first->second, &ins.first->first};
        }
    // The loop over units suits a set whose elements gain more by their unit
    // code than those without one lose by their out-of-line calls; the other
    // sets run general code in the element loop.  On 64 / 300,000 particles,
    // us a turn, general code against units: 100 quadrupoles that are off
    // 111 / 310 against 186 / 493, 100 cavities 135 / 398 against 219 / 631,
    // 100 RF multipoles 1016 / 3702 against 1165 / 5059; 60 quadrupoles that
    // are off among 60 that are on 278 / 895 against 215 / 710, 108 thin kicks
    // with 12 rotated ones 61 / 194 against 47 / 151.
    cs.units = with_units && gain >= 0;
    // A structure that the set holds with many different constants (the
    // bends of ring variants with different cell counts) gets one structure
    // function rather than a literal copy per constant set.
    std::vector<std::pair<Literal *, const std::string *>> ranked;
    for (auto &kv : lits) {
        Literal &v = kv.second;
        if (!all_literal &&
            (v.uses < 2 || lits_of_struct[counted(structs[v.structure])] > kLiteralPerStruct))
            continue;
        if (!all_literal && !write(v)) return cannot(v.line, v.pc);
        ranked.emplace_back(&v, &kv.first);
    }
    std::stable_sort(ranked.begin(), ranked.end(), [](const auto &x, const auto &y) {
        return x.first->uses != y.first->uses ? x.first->uses > y.first->uses
               : x.first->general != y.first->general ? x.first->general < y.first->general
                                                       : x.first->unit < y.first->unit;
    });
    if ((int64_t)ranked.size() > kLiteralMax) ranked.resize(kLiteralMax);
    std::map<const std::string *, int32_t> fn_of_lit;       // by the key in lits
    for (auto &r : ranked) {
        fn_of_lit.emplace(r.second, (int32_t)cs.body.size());
        cs.body.push_back(r.first->general);
        cs.fast.push_back(r.first->unit);
        cs.small.push_back(structs[r.first->structure].small);
    }
    // the other records: structure functions, and the records of each
    std::map<int32_t, int32_t> fn_of_struct;
    std::map<int32_t, std::vector<std::pair<size_t, int64_t>>> records_of;
    recs.assign(nl, {});
    for (size_t l = 0; l < nl; l++) {
        std::map<int64_t, int32_t> fn_of_pc;
        for (auto &pr : record[l]) {
            auto it = fn_of_lit.find(pr.second.second);
            if (it != fn_of_lit.end()) {
                fn_of_pc.emplace(pr.first, it->second);
                continue;
            }
            auto ins = fn_of_struct.emplace(pr.second.first, (int32_t)cs.body.size());
            if (ins.second) {
                cs.body.push_back(structs[pr.second.first].general);
                cs.fast.push_back(structs[pr.second.first].unit);
                cs.small.push_back(0);
            }
            fn_of_pc.emplace(pr.first, ins.first->second);
            records_of[ins.first->second].emplace_back(l, pr.first);
        }
        if ((int64_t)cs.body.size() > XT_CODEGEN_MAX_RECORDS) {
            err = "the code needs more than " + std::to_string(XT_CODEGEN_MAX_RECORDS) +
                  " element functions";
            return XTM_ERR_UNSUPPORTED;
        }
        const std::vector<int64_t> &entry = *entries[l];
        recs[l].resize(entry.size());
        for (size_t e = 0; e < entry.size(); e++) recs[l][e] = fn_of_pc[entry[e]];
    }
    // Constants that all records of a structure share become literals of its
    // unit code: bends with their own field errors load 5 words instead of
    // 150, and a wave alone on its SIMD waits for the scalar loads of each
    // element.  Error ring, 64,000 particles, one turn: 11.7 -> 8.8 ms.
    for (auto &kv : records_of) {
        const size_t l0 = kv.second[0].first;
        const int64_t pc0 = kv.second[0].second;
        std::vector<char> shared;
        for (int64_t k : loaded_words(cs.fast[kv.first])) {
            if (k >= (int64_t)shared.size()) shared.resize(k + 1, 0);
            shared[k] = 1;
        }
        for (size_t k = 0; k < shared.size(); k++)
            for (auto &rc : kv.second)
                shared[k] = shared[k] && wbits((*progs[rc.first])[rc.second + k]) ==
                                             wbits((*progs[l0])[pc0 + k]);
        FastGen f(*progs[l0], true, &shared);
        cs.fast[kv.first] = unit(f, pc0);
    }

    // Segments: runs of consecutive cheap literal records (drifts,
    // apertures, thin kicks, markers) cut into chunks of at most kSegMax
    // elements; a chunk sequence becomes one function that tracks the
    // chunk's elements in order and returns the position of the element where
    // the particle was lost.  The
    // key of a chunk's first element carries the segment number and the
    // chunk length; the loop runs the chunk with one dispatch instead of one
    // per element.  Same element calls, same order: the arithmetic is that
    // of the single-record path.  (Cheap records are literal: their code
    // reads no constants through rp, which the segment call passes for the
    // chunk's first element only.)
    //
    // Where a run is cut decides how often its chunks repeat: pieces of a
    // fixed length suit a run whose period divides it (five cells of six
    // elements), pieces that begin at one record suit runs with irregular
    // parts between like cells.  Lengths and the most frequent records are
    // tried on the whole set, and the cut that leaves the fewest
    // dispatches is kept.  Chunks that occur once are kept only up to
    // kSegOnceBody elements of code.
    using Chunk = std::tuple<size_t, size_t, size_t>;   // (line, first element, length)
    auto cut = [&](size_t len, int32_t head) {
        std::vector<Chunk> out;
        for (size_t l = 0; l < nl; l++) {
            const std::vector<int32_t> &rv = recs[l];
            size_t e = 0;
            while (e < rv.size()) {
                if (!cs.small[rv[e]]) { e++; continue; }
                size_t f = e;
                while (f < rv.size() && cs.small[rv[f]]) f++;
                while (e < f) {
                    size_t n = 1;
                    while (e + n < f && n < len && rv[e + n] != head) n++;
                    if (n > 1) out.emplace_back(l, e, n);
                    e += n;
                }
            }
        }
        return out;
    };
    auto chunk_seq = [&](const Chunk &ch) {
        const std::vector<int32_t> &rv = recs[std::get<0>(ch)];
        return std::vector<int32_t>(rv.begin() + std::get<1>(ch),
                                    rv.begin() + std::get<1>(ch) + std::get<2>(ch));
    };
    using Ranked = std::vector<std::pair<int64_t, std::vector<int32_t>>>;
    // the segments of a cut, best first, and the dispatches that they save
    auto choose = [&](const std::vector<Chunk> &chunks, Ranked &kept) {
        std::map<std::vector<int32_t>, int64_t> count;
        for (auto &ch : chunks) count[chunk_seq(ch)]++;
        Ranked rank;
        for (auto &kv : count)
            rank.emplace_back((kv.second - (kv.second > 1 ? 0 : 1)) * (int64_t)kv.first.size(),
                              kv.first);
        std::stable_sort(rank.begin(), rank.end(), [](const auto &x, const auto &y) {
            return x.first > y.first || (x.first == y.first && x.second.size() > y.second.size());
        });
        int64_t body = 0, saved = 0;
        kept.clear();
        for (auto &r : rank) {
            const int64_t n = (int64_t)r.second.size(), uses = count[r.second];
            if ((int64_t)kept.size() >= kSegMaxCount ||
                body + n > (uses > 1 ? kSegMaxBody : kSegOnceBody))
                continue;
            body += n;
            saved += uses * (n - 1);
            kept.push_back(r);
        }
        // among equal savings, less code
        return saved * 4096 - body;
    };
    std::map<int32_t, int64_t> small_uses;
    int64_t n_small = 0;
    for (auto &rv : recs)
        for (int32_t r : rv)
            if (cs.small[r]) {
                small_uses[r]++;
                n_small++;
            }
    std::vector<std::pair<int64_t, int32_t>> heads;
    for (auto &kv : small_uses) heads.emplace_back(-kv.second, kv.first);
    std::sort(heads.begin(), heads.end());
    if (heads.size() > 16) heads.resize(16);
    std::vector<Chunk> chunks;
    Ranked seg_rank;
    int64_t best = -1;
    auto attempt = [&](size_t len, int32_t head) {
        std::vector<Chunk> c = cut(len, head);
        Ranked kept;
        const int64_t v = choose(c, kept);
        if (v > best) {
            best = v;
            chunks = std::move(c);
            seg_rank = std::move(kept);
        }
    };
    int64_t tries = 4000000 / std::max<int64_t>(n_small, 1);   // bounds the search for long lines
    attempt(kSegMax, -1);
    for (size_t k = 0; k < heads.size() && tries-- > 0; k++) attempt(kSegMax, heads[k].second);
    for (size_t len = kSegMax - 1; len >= 8 && tries-- > 0; len--) attempt(len, -1);
    std::map<std::vector<int32_t>, Chunk> where;
    for (auto &ch : chunks) where.emplace(chunk_seq(ch), ch);
    std::map<std::vector<int32_t>, int32_t> seg_id;
    for (auto &r : seg_rank) {
        seg_id.emplace(r.second, (int32_t)cs.segs.size());
        cs.segs.push_back(r.second);
        const Chunk &ch = where[r.second];
        FastGen f(*progs[std::get<0>(ch)], false);
        for (size_t j = 0; with_units && j < std::get<2>(ch); j++)
            f.direct |= !f.record((*entries[std::get<0>(ch)])[std::get<1>(ch) + j]);
        cs.fast_segs.push_back(f.body());
    }
    for (auto &ch : chunks) {
        auto it = seg_id.find(chunk_seq(ch));
        if (it == seg_id.end()) continue;
        recs[std::get<0>(ch)][std::get<1>(ch)] |= ((it->second + 1) << XT_KEY_SEG_SHIFT) |
                                                  ((int32_t)std::get<2>(ch) << XT_KEY_SPAN_SHIFT);
    }
    return XTM_OK;
}

/* The code set for tracking: with units where it compiles with them and gains
   by them.  Functions are shared by records whose general and unit code
   agree, so a set near XT_CODEGEN_MAX_RECORDS functions may fit without units
   only. */
int choose_code_set(const std::vector<const std::vector<int64_t> *> &entries,
                    const std::vector<const std::vector<double> *> &progs, bool keyed_pc,
                    CodeSet &cs, std::vector<std::vector<int32_t>> &recs, std::string &err) {
    const int st = build_code_set(entries, progs, keyed_pc, true, cs, recs, err);
    if (st == XTM_OK && cs.units) return st;
    if (st != XTM_OK && st != XTM_ERR_UNSUPPORTED) return st;
    return build_code_set(entries, progs, keyed_pc, false, cs, recs, err);
}

/* The functions, segments and element runner of a code set, in namespace
   xt_gen. */
std::string emit_code_set(const CodeSet &cs, uint32_t options, const char *what) {
    const size_t n_fast = cs.units ? cs.fast.size() : 0;
    const size_t n_fast_segs = cs.units ? cs.fast_segs.size() : 0;
    std::string s;
    s += std::string("// generated ") + what + ": element records as straight-line calls\n";
    if (options & XTM_SPEC_FAST_ARITH) s += "#define XTM_ARITH_FAST 1\n";
    s += "#if defined(__HIPCC__) && !defined(__HIPCC_RTC__)\n#include <hip/hip_runtime.h>\n#endif\n";
    s += "#include \"xt_fast.h\"\n\n";
    s += "#if defined(__HIPCC__)\n#define XT_GEN_FN static __host__ __device__ __forceinline__\n";
    s += "#else\n#define XT_GEN_FN static inline\n#endif\n\n";
    s += "namespace xt_gen {\n";
    for (size_t r = 0; r < cs.body.size(); r++) {
        s += "XT_GEN_FN void rec_" + std::to_string(r) +
             "(xt::PState<double> &p, const xt::PRef &m, const double *__restrict__ prog,\n"
             "    xt::CProg rp, const xt::TrackCtx &c) {\n"
             "    (void)m; (void)prog; (void)rp; (void)c;\n";
        s += cs.body[r];
        s += "}\n\n";
    }
    for (size_t r = 0; r < n_fast; r++)
        s += "XT_GEN_FN void fast_" + std::to_string(r) +
             "(xt::FState &p, xt::CProg rp) {\n    (void)p; (void)rp;\n" + cs.fast[r] + "}\n\n";
    for (size_t q = 0; q < n_fast_segs; q++)
        s += "XT_GEN_FN void fast_seg_" + std::to_string(q) + "(xt::FState &p) {\n    (void)p;\n" +
             cs.fast_segs[q] + "}\n\n";
    // a segment's records that address the program (relative literal code
    // of thin kicks: the literal kick's descriptor) get their own element's
    // rp from ent, the entry offsets from the chunk's first element on
    for (size_t q = 0; q < cs.segs.size(); q++) {
        s += "XT_GEN_FN int32_t seg_" + std::to_string(q) +
             "(xt::PState<double> &p, const xt::PRef &m, const double *__restrict__ prog,\n"
             "    xt::CProg rp, const xt::TrackCtx &c, xt::CP<int64_t> ent) {\n"
             "    (void)ent;\n";
        const auto &v = cs.segs[q];
        for (size_t j = 0; j < v.size(); j++) {
            const std::string &b = cs.body[v[j]];
            const bool own_rp = cs.keyed_pc && (b.find("rp[") != std::string::npos ||
                                                b.find("rp + ") != std::string::npos);
            s += "    rec_" + std::to_string(v[j]) + "(p, m, prog, " +
                 (own_rp ? "xt::cptr(prog) + ent[" + std::to_string(j) + "]" : std::string("rp")) +
                 ", c);";
            s += j + 1 < v.size() ? " if (p.state <= 0) return " + std::to_string(j) + ";\n"
                                  : " return " + std::to_string(j) + ";\n";
        }
        s += "}\n\n";
    }
    // element key: the function index with the segment fields (int32), and
    // with relative addressing also the element's program offset
    const std::string kr = cs.keyed_pc ? "xt::uniform(k.r)" : "xt::uniform(k)";
    s += "struct Runner {\n"
         "    const int32_t *__restrict__ rec;\n"
         "    const int64_t *__restrict__ entry;\n"
         "    const double *__restrict__ prog;\n";
    s += "    static constexpr bool kSegments = true;\n";
    if (cs.keyed_pc)
        s += "    struct Key { int32_t r; int64_t pc; };\n"
             "    XT_HD Key key(int64_t e) const { return Key{xt::cptr(rec)[e], xt::cptr(entry)[e]}; }\n";
    else
        s += "    using Key = int32_t;\n"
             "    XT_HD Key key(int64_t e) const { return xt::cptr(rec)[e]; }\n";
    const std::string rp = cs.keyed_pc
                               ? "        const xt::CProg rp = xt::cptr(prog) + xt::uniform(k.pc);\n"
                               : "        const xt::CProg rp = xt::cptr(prog);\n";
    s += "    XT_HD static int32_t span(Key k) { return (" + kr + " >> " +
         std::to_string(XT_KEY_SPAN_SHIFT) + ") & " + std::to_string(XT_KEY_SPAN_MASK) +
         "; }\n"
         "    XT_HD int32_t segment(xt::PState<double> &p, const xt::PRef &m, Key k,\n"
         "                          const xt::TrackCtx &c, int64_t e) const {\n" + rp +
         "        const xt::CP<int64_t> ent = xt::cptr(entry) + xt::uniform(e);\n"
         "        switch (" + kr + " >> " + std::to_string(XT_KEY_SEG_SHIFT) + ") {\n";
    for (size_t q = 0; q < cs.segs.size(); q++)
        s += "        case " + std::to_string(q + 1) + ": return seg_" + std::to_string(q) +
             "(p, m, prog, rp, c, ent);\n";
    s += "        default: p.state = -999; return 0;\n"
         "        }\n"
         "    }\n"
         "    XT_HD void operator()(xt::PState<double> &p, const xt::PRef &m, Key k,\n"
         "                          const xt::TrackCtx &c) const {\n" + rp +
         "        switch (" + kr + " & " + std::to_string(XT_KEY_REC_MASK) + ") {\n";
    for (size_t r = 0; r < cs.body.size(); r++)
        s += "        case " + std::to_string(r) + ": rec_" + std::to_string(r) +
             "(p, m, prog, rp, c); break;\n";
    s += "        default: p.state = -999; break;\n"
         "        }\n"
         "    }\n";
    if (cs.units) {
        s += "    /* the units of xt_fast.h */\n"
             "    XT_HD void fast_segment(xt::FState &p, Key k) const {\n"
             "        switch (" + kr + " >> " + std::to_string(XT_KEY_SEG_SHIFT) + ") {\n";
        for (size_t q = 0; q < n_fast_segs; q++)
            s += "        case " + std::to_string(q + 1) + ": fast_seg_" + std::to_string(q) +
                 "(p); break;\n";
        s += "        default: p.bad = true; break;\n"
             "        }\n"
             "    }\n"
             "    XT_HD void fast(xt::FState &p, Key k) const {\n" + rp +
             "        switch (" + kr + " & " + std::to_string(XT_KEY_REC_MASK) + ") {\n";
        for (size_t r = 0; r < n_fast; r++)
            s += "        case " + std::to_string(r) + ": fast_" + std::to_string(r) +
                 "(p, rp); break;\n";
        s += "        default: p.bad = true; break;\n"
             "        }\n"
             "    }\n";
    }
    s += "};\n";
    return s;
}

}  // namespace

namespace {

/* The call that tracks the chi == 1 particle i of a kernel (device) or of the
   host build: with the loop over units every lane of a wave takes part. */
std::string track_call(bool units, bool backtrack, bool device, const std::string &pad,
                       const std::string &runner, const std::string &args) {
    const std::string in = "\n" + pad + "    ";
    if (units)
        return pad + "xt::track_particle_units<" + (backtrack ? "true" : "false") + ">(" +
               (device ? "P" : "*P") + ", i, " + (device ? "alive" : "true") + "," + in + runner +
               ", c," + in + args + ", " + (device ? "xt::kernarg()" : "mon") + ");\n";
    return (device ? pad + "const xt::MonRef mon = xt::kernarg();\n" + pad + "if (alive)\n    "
                   : std::string()) +
           pad + "xt::track_particle_loop<true, false>(" + (device ? "*mon.P" : "*P") + ", i," +
           in + runner + ", c," + in + args + ", mon);\n";
}

int line_source(const std::vector<int64_t> &entry, const std::vector<double> &prog,
                int32_t waves_per_eu, uint32_t options, std::string &src,
                std::vector<int32_t> &rec_of_elem, std::string &err, bool backtrack) {
    CodeSet cs;
    std::vector<std::vector<int32_t>> recs;
    // backwards there is no loop over compiled general code
    const int st = backtrack
                       ? build_code_set({&entry}, {&prog}, false, true, cs, recs, err)
                       : choose_code_set({&entry}, {&prog}, false, cs, recs, err);
    if (st != XTM_OK) return st;
    if (backtrack) cs.units = true;
    rec_of_elem = std::move(recs[0]);
    std::string s = emit_code_set(cs, options, "line code");
    const std::string run = "xt_gen::Runner{rec, entry, prog}";
    const std::string args = "num_turns, ele_start, num_ele_track, flag_end_turn_actions, "
                             "flag_reset_s, flag_monitor";
    s += "}  // namespace xt_gen\n\n";
    s += "#if defined(__HIPCC__)\n";
    char occ[128];
    std::snprintf(occ, sizeof occ, "__attribute__((amdgpu_waves_per_eu(%d)))",
                  waves_per_eu > 0 ? waves_per_eu : 1);
    s += std::string("extern \"C\" __global__ __launch_bounds__(256) ") +
         (waves_per_eu > 0 ? occ : "") +
         "\nvoid xtm_line_kernel(xtm_particles P, xtm_monitor M, xtm_features F,\n"
         "    const int32_t *__restrict__ rec, const int64_t *__restrict__ entry, const double *__restrict__ prog,\n"
         "    double line_length, int32_t num_turns, int32_t ele_start, int32_t num_ele_track,\n"
         "    int32_t flag_end_turn_actions, int32_t flag_reset_s, int32_t flag_monitor,\n"
         "    uint64_t flags, int32_t num_ele_line) {\n"
         "    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;\n"
         "    const xt::TrackCtx c{flags, line_length, P.q0, P.t_sim, num_ele_line};\n"
         "    // chi == 1 particles; the interpreter kernel tracks the others\n"
         "    const bool alive = i < P.capacity && P.state[i] > 0 && P.chi[i] == 1.0;\n" +
         track_call(cs.units, backtrack, true, "    ", run, args) +
         "}\n"
         "#else\n"
         "// host build (tests): the same per-particle body over all particles\n"
         "extern \"C\" void xtm_line_host(const int32_t *rec, const int64_t *entry, const double *prog,\n"
         "    double line_length, const xtm_particles *P, int32_t num_turns, int32_t ele_start,\n"
         "    int32_t num_ele_track, int32_t flag_end_turn_actions, int32_t flag_reset_s,\n"
         "    int32_t flag_monitor, const xtm_monitor *M, uint64_t flags) {\n"
         "    xtm_monitor m0 = {};\n" +
         (backtrack ? std::string("    const int64_t num_ele_line = ") +
                          std::to_string(entry.size()) + ";\n"
                    : std::string("    const int64_t num_ele_line = 0;\n")) +
         "    const xt::TrackCtx c{flags, line_length, P->q0, P->t_sim, num_ele_line};\n"
         "    const xt::MonRef mon{M ? M : &m0, P};\n"
         "    for (int64_t i = 0; i < P->capacity; i++) {\n"
         "        if (!(P->state[i] > 0)) continue;\n"
         "        if (P->chi[i] == 1.0)\n" +
         track_call(cs.units, backtrack, false, "            ", run, args) +
         "        else\n"
         "            xt::track_particle_loop_cold<false>(*P, i, xt::ProgramRunner{entry, prog},\n"
         "                c, " + args + ", mon);\n"
         "    }\n"
         "}\n"
         "#endif\n";
    src = std::move(s);
    return XTM_OK;
}

}  // namespace

int xt_generate_line_source(const std::vector<int64_t> &entry, const std::vector<double> &prog,
                            int32_t waves_per_eu, uint32_t options, std::string &src,
                            std::vector<int32_t> &rec_of_elem, std::string &err) {
    return line_source(entry, prog, waves_per_eu, options, src, rec_of_elem, err, false);
}

bool xt_source_has_units(const std::string &src) {
    return src.find("xt::track_particle_units") != std::string::npos;
}

int xt_generate_backtrack_source(const std::vector<int64_t> &entry,
                                 const std::vector<double> &prog, int32_t waves_per_eu,
                                 std::string &src, std::vector<int32_t> &rec_of_elem,
                                 std::string &err) {
    return line_source(entry, prog, waves_per_eu, 0, src, rec_of_elem, err, true);
}


int xt_generate_batch_source(const std::vector<const std::vector<int64_t> *> &entries,
                             const std::vector<const std::vector<double> *> &progs,
                             int32_t waves_per_eu, std::string &src,
                             std::vector<std::vector<int32_t>> &recs, std::string &err) {
    CodeSet cs;
    // the batch kernel's runner reads each element's program offset
    const int st = choose_code_set(entries, progs, true, cs, recs, err);
    if (st != XTM_OK) return st;
    std::string s = emit_code_set(cs, 0, "batch code");
    s += "/* one block of a batch: particles [first, first + count) of line `line` */\n"
         "struct BatchBlock { int64_t first; int32_t line; int32_t count; };\n"
         "}  // namespace xt_gen\n\n";
    char occ[128];
    std::snprintf(occ, sizeof occ, "__attribute__((amdgpu_waves_per_eu(%d)))",
                  waves_per_eu > 0 ? waves_per_eu : 1);
    s += "#if defined(__HIPCC__)\n";
    s += std::string("extern \"C\" __global__ __launch_bounds__(256) ") +
         (waves_per_eu > 0 ? occ : "") +
         "\nvoid xtm_batch_line_kernel(xtm_particles P, xtm_monitor M, xtm_features F,\n"
         "    int32_t flag_monitor, const xt_gen::BatchBlock *__restrict__ blocks,\n"
         "    const int32_t *const *__restrict__ recs, const int64_t *const *__restrict__ entries,\n"
         "    const double *const *__restrict__ progs, const int64_t *__restrict__ nele,\n"
         "    const double *__restrict__ lengths, int32_t num_turns, uint64_t flags) {\n"
         "    const xt_gen::BatchBlock b = xt::cptr(blocks)[blockIdx.x];\n"
         "    const int64_t i = b.first + threadIdx.x;\n"
         "    const int64_t ne = xt::cptr(nele)[b.line];\n"
         "    const xt::TrackCtx c{flags, xt::cptr(lengths)[b.line], P.q0, P.t_sim, ne};\n"
         "    // chi == 1 particles; the interpreter batch kernel tracks the others\n"
         "    const bool alive = (int32_t)threadIdx.x < b.count && P.state[i] > 0 &&\n"
         "                       P.chi[i] == 1.0;\n" +
         track_call(cs.units, false, true, "    ",
                    "xt_gen::Runner{xt::cptr(recs)[b.line], xt::cptr(entries)[b.line], "
                    "xt::cptr(progs)[b.line]}",
                    "num_turns, 0, (int32_t)ne, 1, 1, flag_monitor") +
         "}\n"
         "#else\n"
         "// host build (tests): the same per-particle body over the blocks\n"
         "extern \"C\" void xtm_batch_host(const xt_gen::BatchBlock *blocks, int64_t num_blocks,\n"
         "    const int32_t *const *recs, const int64_t *const *entries, const double *const *progs,\n"
         "    const int64_t *nele, const double *lengths, const xtm_particles *P,\n"
         "    int32_t num_turns, uint64_t flags) {\n"
         "    for (int64_t bi = 0; bi < num_blocks; bi++) {\n"
         "        const xt_gen::BatchBlock b = blocks[bi];\n"
         "        const int64_t ne = nele[b.line];\n"
         "        const xt::TrackCtx c{flags, lengths[b.line], P->q0, P->t_sim, ne};\n"
         "        const xt::MonRef mon{nullptr, P};\n"
         "        for (int64_t i = b.first; i < b.first + b.count; i++) {\n"
         "            if (!(P->state[i] > 0)) continue;\n"
         "            if (P->chi[i] == 1.0)\n" +
         track_call(cs.units, false, false, "                ",
                    "xt_gen::Runner{recs[b.line], entries[b.line], progs[b.line]}",
                    "num_turns, 0, (int32_t)ne, 1, 1, 0") +
         "            else\n"
         "                xt::track_particle_loop_cold<false>(*P, i,\n"
         "                    xt::ProgramRunner{entries[b.line], progs[b.line]}, c, num_turns, 0,\n"
         "                    (int32_t)ne, 1, 1, 0, mon);\n"
         "        }\n"
         "    }\n"
         "}\n"
         "#endif\n";
    src = std::move(s);
    return XTM_OK;
}
