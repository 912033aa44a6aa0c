// hamr_adjoint.h -- hand-written reverse-mode derivatives of the pointwise
// physics of one forward stage (FP64): the MHD state and fluxes of a
// reconstructed face state, the HLL combination, the cell-centre EMF, and the
// PPM reconstruction through the limiter's active branch.  Every function
// recomputes the primal quantities it needs from its inputs (nothing of the
// forward pass is stored).
//
// Conventions follow hamr_phys.h: prims RHO, UU, U1-U3 (relative 4-velocity),
// B1-B3, KTOT; packed symmetric metric; fluxes and conserved variables times
// gdet.  Branch points (the clamps of gamma_calc and of the magnetosonic speed,
// the max/min of the HLL speeds, the limiter's cases) take the derivative of the
// branch the primal takes.
#pragma once

#include "hamr_phys.h"

namespace hamr {

// the double versions stay visible beside the Dual overloads below
using ::copysign;
using ::fabs;
using ::fmin;

// ---------------------------------------------------------------------------
// Forward-mode number with N tangents (PPM Jacobian w.r.t. its 5 inputs).  The Jacobian
// forms, up to para_jacobian, are in no kernel: the host checks hold para_vjp, which
// is, against them.
template <int N> struct Dual {
    double v, d[N];
    HD Dual() : v(0.) { for (int k = 0; k < N; k++) d[k] = 0.; }
    HD Dual(double x) : v(x) { for (int k = 0; k < N; k++) d[k] = 0.; }
};
template <int N> HD Dual<N> operator+(const Dual<N> &a, const Dual<N> &b)
{ Dual<N> r; r.v = a.v + b.v; for (int k = 0; k < N; k++) r.d[k] = a.d[k] + b.d[k]; return r; }
template <int N> HD Dual<N> operator-(const Dual<N> &a, const Dual<N> &b)
{ Dual<N> r; r.v = a.v - b.v; for (int k = 0; k < N; k++) r.d[k] = a.d[k] - b.d[k]; return r; }
template <int N> HD Dual<N> operator-(const Dual<N> &a)
{ Dual<N> r; r.v = -a.v; for (int k = 0; k < N; k++) r.d[k] = -a.d[k]; return r; }
template <int N> HD Dual<N> operator*(const Dual<N> &a, const Dual<N> &b)
{ Dual<N> r; r.v = a.v * b.v; for (int k = 0; k < N; k++) r.d[k] = a.d[k] * b.v + a.v * b.d[k]; return r; }
// The value is the IEEE quotient; the tangents use one reciprocal of b (an
// FP64 division per tangent would cost as much as the rest of the parabola).
template <int N> HD Dual<N> operator/(const Dual<N> &a, const Dual<N> &b)
{
    Dual<N> r;
    r.v = a.v / b.v;
    const double ib = 1. / b.v;
    for (int k = 0; k < N; k++) r.d[k] = (a.d[k] - r.v * b.d[k]) * ib;
    return r;
}
template <int N> HD bool operator<(const Dual<N> &a, const Dual<N> &b) { return a.v < b.v; }
template <int N> HD bool operator>(const Dual<N> &a, const Dual<N> &b) { return a.v > b.v; }
template <int N> HD bool operator<=(const Dual<N> &a, const Dual<N> &b) { return a.v <= b.v; }
template <int N> HD Dual<N> fabs(const Dual<N> &a) { return (a.v < 0.) ? -a : a; }
template <int N> HD Dual<N> fmin(const Dual<N> &a, const Dual<N> &b) { return (b.v < a.v) ? b : a; }
template <int N> HD Dual<N> copysign(const Dual<N> &a, const Dual<N> &s)
{
    const bool neg = __builtin_signbit(s.v), aneg = __builtin_signbit(a.v);
    return (neg == aneg) ? a : -a;
}
template <int N> HD Dual<N> dv(Dual<N> a, Dual<N> b) { return a / b; }

// d(l, r)/d(x1..x5) of para for one cell: Jl[5], Jr[5] (forward mode over
// all five inputs; the reference form of para_jacobian below).
HD void para_jacobian_dual(const double *x, double *l, double *r, double *Jl, double *Jr)
{
    Dual<5> y[5];
    for (int k = 0; k < 5; k++) {
        y[k] = Dual<5>(x[k]);
        y[k].d[k] = 1.;
    }
    Dual<5> lo, ro;
    para(y[0], y[1], y[2], y[3], y[4], lo, ro);
    *l = lo.v;
    *r = ro.v;
    for (int k = 0; k < 5; k++) {
        Jl[k] = lo.d[k];
        Jr[k] = ro.d[k];
    }
}

// Tangent of mc_slope(ym, y0, yp) along the branch it takes (the choices of
// para_jacobian_dual's fabs, fmin and copysign): s * dX, X the selected one of
// Dqm = 2 (y0 - ym), Dqp = 2 (yp - y0), Dqc = 0.5 (yp - ym); t over (ym, y0, yp).
HD void mc_slope_tangent(double ym, double y0, double yp, double t[3])
{
    const double Dqm = 2. * (y0 - ym), Dqp = 2. * (yp - y0), Dqc = 0.5 * (yp - ym);
    t[0] = t[1] = t[2] = 0.;
    if (!(Dqm * Dqp > 0.)) return;
    const double am = fabs(Dqm), ap = fabs(Dqp), ac = fabs(Dqc);
    const bool pick_p = ap < am;                // fmin(|Dqm|, |Dqp|)
    const double m = pick_p ? ap : am;
    const double sgn = __builtin_signbit(Dqc) ? -1. : 1.;  // copysign(., Dqc) of a positive value
    if (m < ac) {
        if (pick_p) {
            const double f = sgn * (Dqp < 0. ? -2. : 2.);
            t[1] = -f;
            t[2] = f;
        } else {
            const double f = sgn * (Dqm < 0. ? -2. : 2.);
            t[0] = -f;
            t[1] = f;
        }
    } else {
        const double f = sgn * (Dqc < 0. ? -0.5 : 0.5);
        t[0] = -f;
        t[2] = f;
    }
}

// d(l, r)/d(x1..x5) of para for one cell: Jl[5], Jr[5], in closed form along
// the limiter's active branches (the slopes' tangents have three entries, the
// interface values' four): the values are para's; the tangents equal
// para_jacobian_dual's up to the rounding of the division by 6.
HD void para_jacobian(const double *x, double *l, double *r, double *Jl, double *Jr)
{
    double dq[3], t[3][5];
    for (int s = 0; s < 3; s++) {
        dq[s] = mc_slope(x[s], x[s + 1], x[s + 2]);
        double ts[3];
        mc_slope_tangent(x[s], x[s + 1], x[s + 2], ts);
        for (int k = 0; k < 5; k++) t[s][k] = (k >= s && k < s + 3) ? ts[k - s] : 0.;
    }
    const double sixth = 1. / 6.;
    // interface values below and above cell x3 (ppm_face) and their tangents
    double lo = ppm_face(x[1], x[2], dq[0], dq[1]), hi = ppm_face(x[2], x[3], dq[1], dq[2]);
    double tl[5], tr[5];
    for (int k = 0; k < 5; k++) {
        tl[k] = 0.5 * ((k == 2 ? 1. : 0.) + (k == 1 ? 1. : 0.)) - (t[1][k] - t[0][k]) * sixth;
        tr[k] = 0.5 * ((k == 3 ? 1. : 0.) + (k == 2 ? 1. : 0.)) - (t[2][k] - t[1][k]) * sixth;
    }
    // ppm_limit on values and tangents
    const double x3 = x[2];
    const double qa = (hi - x3) * (x3 - lo), qd = hi - lo, qe = 6.0 * (x3 - 0.5 * (lo + hi));
    if (qa <= 0.) {
        lo = x3;
        hi = x3;
        for (int k = 0; k < 5; k++) tl[k] = tr[k] = (k == 2 ? 1. : 0.);
    }
    if (qd * (qd - qe) < 0.) {
        lo = 3.0 * x3 - 2.0 * hi;
        for (int k = 0; k < 5; k++) tl[k] = 3.0 * (k == 2 ? 1. : 0.) - 2.0 * tr[k];
    } else if (qd * (qd + qe) < 0.) {
        hi = 3.0 * x3 - 2.0 * lo;
        for (int k = 0; k < 5; k++) tr[k] = 3.0 * (k == 2 ? 1. : 0.) - 2.0 * tl[k];
    }
    *l = lo;
    *r = hi;
    for (int k = 0; k < 5; k++) {
        Jl[k] = tl[k];
        Jr[k] = tr[k];
    }
}

// mc_slope(ym, y0, yp) with the choice it makes: the slope is 2 (y0 - ym), 2 (yp -
// y0) or (yp - ym) / 2 itself, as the three agree in sign where it is not zero.
struct SlopeChoice {
    double dq;
    bool on, centred, upper;
    HD SlopeChoice(double ym, double y0, double yp)
    {
        const double Dqm = 2. * (y0 - ym), Dqp = 2. * (yp - y0), Dqc = 0.5 * (yp - ym);
        on = Dqm * Dqp > 0.;
        upper = fabs(Dqp) < fabs(Dqm);
        const double one_sided = upper ? Dqp : Dqm;
        centred = !(fabs(one_sided) < fabs(Dqc));
        dq = on ? (centred ? Dqc : one_sided) : 0.;
    }
    // adds lam d(dq)/d(ym, y0, yp) to v[0..2]
    HD void vjp(double lam, double *v) const
    {
        const double h = on ? (centred ? 0.5 : 2.) * lam : 0.;
        const double lo = !centred && upper ? 0. : h, hi = centred || upper ? h : 0.;
        v[0] -= lo;
        v[1] += lo - hi;
        v[2] += hi;
    }
};

// Reverse of para for one cell: adds lam_l dl/dx + lam_r dr/dx to v[0..4], along
// the branches para_jacobian takes.
HD void para_vjp(const double *x, double ll, double lr, double *v)
{
    const SlopeChoice s0(x[0], x[1], x[2]), s1(x[1], x[2], x[3]), s2(x[2], x[3], x[4]);
    const double x3 = x[2];
    const double lo = ppm_face(x[1], x3, s0.dq, s1.dq), hi = ppm_face(x3, x[3], s1.dq, s2.dq);
    const double qa = (hi - x3) * (x3 - lo), qd = hi - lo, qe = 6.0 * (x3 - 0.5 * (lo + hi));
    const bool low = qd * (qd - qe) < 0., high = !low && qd * (qd + qe) < 0., flat = qa <= 0.;
    // low: l = 3 x3 - 2 r, high: r = 3 x3 - 2 l
    const double fl = low ? 0. : high ? ll - 2.0 * lr : ll, fr = high ? 0. : low ? lr - 2.0 * ll : lr;
    const double l3 = low ? 3.0 * ll : high ? 3.0 * lr : 0.;
    // flat: l = r = x3, else the interface values
    const double gl = flat ? 0. : 0.5 * fl, gr = flat ? 0. : 0.5 * fr, third = 1. / 3.;
    v[1] += gl;
    v[2] += l3 + (flat ? fl + fr : gl + gr);
    v[3] += gr;
    s0.vjp(gl * third, v);
    s1.vjp((gr - gl) * third, v + 1);
    s2.vjp(-gr * third, v + 2);
}

// ---------------------------------------------------------------------------
// Adjoints of the MHD state of one set of primitives (ucon, ucov, bcon, bcov,
// rho, u), pulled back to the primitives by state_pullback.
struct StateAdj {
    double ucon[4], ucov[4], bcon[4], bcov[4], rho, u, bsq;
};

// One state's flux along d (0: its conserved variables; primtoflux,
// GPU_phys_mhd.h:432), contracted with weights lf of its nine components that
// hold the factor gdet:
//   S(d) = u^d Q - b^d R + ptot lf_d,
//   Q = rho (lf_rho + lf_u + lf_K entr) + eta lf_j u_j + lf_Bj b^j,  R = lf_j b_j + lf_Bj u^j,
// lf_j the weights of T^d_j.  The HLL adjoint needs no flux by itself, only
// these sums, and its weights of a state's flux and of its conserved variables
// are lf times one number each; so Q, R and their factors serve both.
struct Contraction {
    double eta, ptot, mu, Q, R, rmg, entr, bsq, w;
    HD Contraction(const double *pr, const State<double> &q, double gam, const double *lf)
    {
        const double rho = pr[RHO], u = pr[UU], P = (gam - 1.) * u;
        w = rho + P + u;
        bsq = dot4(q.bcon, q.bcov);
        eta = w + bsq;
        ptot = P + 0.5 * bsq;
        rmg = rpow(rho, -gam);
        entr = P * rmg;
        const double *m = lf + UU, *n = lf + B1;
        mu = dot4(m, q.ucov);
        Q = rho * (lf[RHO] + lf[UU] + lf[KTOT] * entr) + eta * mu
            + (n[0] * q.bcon[1] + n[1] * q.bcon[2] + n[2] * q.bcon[3]);
        R = dot4(m, q.bcov) + (n[0] * q.ucon[1] + n[1] * q.ucon[2] + n[2] * q.ucon[3]);
    }
    HD double S(const State<double> &q, const double *lf, int d) const
    {
        return q.ucon[d] * Q - q.bcon[d] * R + ptot * lf[UU + d];
    }
};
static_assert(U1 == UU + 1 && U2 == UU + 2 && U3 == UU + 3 && B2 == B1 + 1 && B3 == B1 + 2, "order of the components");

// The adjoint of sF S(dir) + sU S(0): sets a.
HD void contraction_vjp(const double *pr, const State<double> &q, const Contraction &c, int dir, double gam,
                        const double *lf, double sF, double sU, StateAdj &a)
{
    const double Wu = sF * q.ucon[dir] + sU * q.ucon[0], Wb = sF * q.bcon[dir] + sU * q.bcon[0];
    const double Wm = sF * lf[UU + dir] + sU * lf[UU];
    const double *m = lf + UU, *n = lf + B1;
    a.ucon[0] = sU * c.Q;
    a.bcon[0] = -sU * c.R;
    for (int j = 1; j < 4; j++) {
        a.ucon[j] = -Wb * n[j - 1];
        a.bcon[j] = Wu * n[j - 1];
    }
    for (int j = 0; j < 4; j++) {
        a.ucov[j] = Wu * c.eta * m[j];
        a.bcov[j] = -Wb * m[j];
    }
    a.ucon[dir] += sF * c.Q;
    a.bcon[dir] -= sF * c.R;
    const double leta = Wu * c.mu;
    a.rho = Wu * (lf[RHO] + lf[UU] + (1. - gam) * lf[KTOT] * c.entr) + leta;
    a.u = Wu * lf[KTOT] * pr[RHO] * (gam - 1.) * c.rmg + leta * gam + Wm * (gam - 1.);
    a.bsq = leta + 0.5 * Wm;
}

// Magnetosonic speeds of a state along dir (vchar_coord, GPU_phys_mhd.h:550-617)
// with what their reverse uses.
struct Speeds {
    double vp, vm, A, B, C, sd, cms2, cs2, va2, Acon_0, Acon_js;
    Div<double> by_w, by_eta, by_2A;
    bool clamped, dclamp;
    HD Speeds(const double *pr, const State<double> &q, const Contraction &c, int dir, const Geom<double> &G, double gam)
        : by_w(c.w), by_eta(c.eta), by_2A(1.)
    {
        if (dir == 1) { Acon_0 = G.gcon[1]; Acon_js = G.gcon[4]; }
        else if (dir == 2) { Acon_0 = G.gcon[2]; Acon_js = G.gcon[7]; }
        else { Acon_0 = G.gcon[3]; Acon_js = G.gcon[9]; }
        cs2 = by_w(gam * (gam - 1.) * pr[UU]);
        va2 = by_eta(c.bsq);
        cms2 = cs2 + va2 - cs2 * va2;
        clamped = false;
        if (cms2 < 0.) { cms2 = kSMALL; clamped = true; }
        if (cms2 > 1.) { cms2 = 1.; clamped = true; }
        const double Bsq = G.gcon[0], Au = q.ucon[dir], Bu = q.ucon[0];
        A = Bu * Bu - (Bsq + Bu * Bu) * cms2;
        B = 2. * (Au * Bu - (Acon_0 + Au * Bu) * cms2);
        C = Au * Au - (Acon_js + Au * Au) * cms2;
        double discr = B * B - 4. * A * C;
        dclamp = !(discr > 0.);
        if (dclamp) discr = 0.;
        sd = sqrt(discr);
        by_2A = Div<double>(2. * A);
        vp = by_2A(B - sd);
        vm = by_2A(B + sd);
    }
    HD double vmax() const { return mymax(vp, vm); }
    HD double vmin() const { return mymin(vp, vm); }

    // adds the adjoint of lvmax vmax + lvmin vmin to a
    HD void vjp(const State<double> &q, int dir, const Geom<double> &G, double gam, double lvmax, double lvmin,
                StateAdj &a) const
    {
        const double lvp = vp > vm ? lvmax : lvmin, lvm = vp > vm ? lvmin : lvmax;
        double lB = by_2A(lvp + lvm), lA = -2. * by_2A(lvp * vp + lvm * vm), lC = 0.;
        if (!dclamp) {
            const double ld = Div<double>(2. * sd)(by_2A(lvm - lvp));
            lB += ld * 2. * B;
            lA += -4. * C * ld;
            lC = -4. * A * ld;
        }
        const double Bsq = G.gcon[0], Au = q.ucon[dir], Bu = q.ucon[0], om = 1. - cms2;
        a.ucon[0] += lA * 2. * Bu * om + lB * 2. * Au * om;
        a.ucon[dir] += lB * 2. * Bu * om + lC * 2. * Au * om;
        if (clamped) return;
        const double lcms2 = -lA * (Bsq + Bu * Bu) - lB * 2. * (Acon_0 + Au * Bu) - lC * (Acon_js + Au * Au);
        const double lw = by_w(lcms2 * (1. - va2)), le = by_eta(lcms2 * (1. - cs2));
        // cs2 = gam (gam - 1) u / w, w = rho + gam u
        a.u += lw * gam * ((gam - 1.) - cs2);
        a.rho -= lw * cs2;
        // va2 = bsq / eta, eta = rho + gam u + bsq
        const double leta = -le * va2;
        a.bsq += le + leta;
        a.rho += leta;
        a.u += leta * gam;
    }
};

// get_state (GPU_phys_mhd.h:692-760), reverse: adds the primitives' adjoints to lpr.
HD void state_pullback(const double *pr, const State<double> &q, const Geom<double> &G, const Lapse<double> &L,
                       StateAdj &a, double *lpr)
{
    // bsq = bcon . bcov
    for (int m = 0; m < 4; m++) {
        a.bcon[m] += a.bsq * q.bcov[m];
        a.bcov[m] += a.bsq * q.bcon[m];
    }
    // bcov = g bcon
    {
        double t[4];
        lower10(a.bcov, G.gcov, t);
        for (int m = 0; m < 4; m++) a.bcon[m] += t[m];
    }
    // bcon[j] = (B_j + b0 u^j) / u0, b0 = B . ucov(1..3)
    const Div<double> by_u0(q.ucon[0]);
    const double b0 = q.bcon[0];
    double lb0 = a.bcon[0];
    for (int j = 1; j < 4; j++) {
        const double l = by_u0(a.bcon[j]);
        lpr[B1 + j - 1] += l;
        lb0 += l * q.ucon[j];
        a.ucon[j] += l * b0;
        a.ucon[0] -= l * q.bcon[j];
    }
    for (int i = 1; i < 4; i++) {
        lpr[B1 + i - 1] += lb0 * q.ucov[i];
        a.ucov[i] += lb0 * pr[B1 + i - 1];
    }
    // ucov = g ucon
    {
        double t[4];
        lower10(a.ucov, G.gcov, t);
        for (int m = 0; m < 4; m++) a.ucon[m] += t[m];
    }
    // ucon[0] = gamma / alpha, ucon[j] = U_j - gamma beta_j / alpha
    double lgam = a.ucon[0];
    for (int j = 1; j < 4; j++) {
        lgam -= a.ucon[j] * L.beta[j];
        lpr[U1 + j - 1] += a.ucon[j];
    }
    lgam = L.by_alpha(lgam);
    // gamma = sqrt(1 + qsq), qsq = U . g_spatial . U (no derivative where clamped)
    const double *g = G.gcov;
    const double U[3] = {pr[U1], pr[U2], pr[U3]};
    const double v0 = g[4] * U[0] + g[5] * U[1] + g[6] * U[2], v1 = g[5] * U[0] + g[7] * U[1] + g[8] * U[2],
                 v2 = g[6] * U[0] + g[8] * U[1] + g[9] * U[2];
    const double qsq = g[4] * U[0] * U[0] + g[7] * U[1] * U[1] + g[9] * U[2] * U[2]
        + 2. * (g[5] * U[0] * U[1] + g[6] * U[0] * U[2] + g[8] * U[1] * U[2]);
    if (qsq >= 0.) {
        const double lq = Div<double>(sqrt(1. + qsq))(lgam);
        lpr[U1] += lq * v0;
        lpr[U2] += lq * v1;
        lpr[U3] += lq * v2;
    }
    lpr[RHO] += a.rho;
    lpr[UU] += a.u;
}

// Conserved variables U(P) (primtoflux, dir 0) with weights lU, and the
// cell-centre EMF E_i = -gdet (u^j b^k - u^k b^j) (GPU_const_trans.h:63-119) with
// weights lE, reverse: sets lpr.
HD void cell_vjp(const double *pr, const Geom<double> &G, double gam, const double *lU, const double *lE, double *lpr)
{
    const Lapse<double> L(G);
    State<double> q;
    get_state(pr, G, L, q);
    double lf[NPR];
    for (int k = 0; k < NPR; k++) {
        lf[k] = G.g * lU[k];
        lpr[k] = 0.;
    }
    const Contraction c(pr, q, gam, lf);
    StateAdj a;
    contraction_vjp(pr, q, c, 0, gam, lf, 0., 1., a);
    const double *u = q.ucon, *b = q.bcon;
    // E1 = -g (u2 b3 - u3 b2), E2 = -g (u3 b1 - u1 b3), E3 = -g (u1 b2 - u2 b1)
    const double l1 = -G.g * lE[0], l2 = -G.g * lE[1], l3 = -G.g * lE[2];
    a.ucon[1] += l3 * b[2] - l2 * b[3];
    a.ucon[2] += l1 * b[3] - l3 * b[1];
    a.ucon[3] += l2 * b[1] - l1 * b[2];
    a.bcon[1] += l2 * u[3] - l3 * u[2];
    a.bcon[2] += l3 * u[1] - l1 * u[3];
    a.bcon[3] += l1 * u[2] - l2 * u[1];
    state_pullback(pr, q, G, L, a, lpr);
}

// HLL flux through a face (nine components with weights lf) of the states pl
// and pr, reverse: sets lpl and lpr.
HD void hll_vjp(const double *pl, const double *pr, const Geom<double> &G, int dir, double gam, double *lf, double *lpl,
                double *lpr)
{
    for (int k = 0; k < NPR; k++) {
        lf[k] *= G.g;
        lpl[k] = lpr[k] = 0.;
    }
    const Lapse<double> L(G);
    State<double> ql, qr;
    get_state(pl, G, L, ql);
    get_state(pr, G, L, qr);
    const Contraction cl(pl, ql, gam, lf), cr(pr, qr, gam, lf);
    const Speeds vl(pl, ql, cl, dir, G, gam), vr(pr, qr, cr, dir, G, gam);
    const double vxl = vl.vmax(), vnl = vl.vmin(), vxr = vr.vmax(), vnr = vr.vmin();
    const double m1 = mymax(0., vxl), cmax = fabs(mymax(m1, vxr));
    const double n1 = mymax(0., -vnl), cmin = fabs(mymax(n1, -vnr));
    const Div<double> by_den(cmax + cmin + kSMALL);
    // reverse of F = (cmax FL + cmin FR - cmax cmin (UR - UL)) / den
    const double SL = cl.S(ql, lf, dir), SR = cr.S(qr, lf, dir), D = cr.S(qr, lf, 0) - cl.S(ql, lf, 0);
    const double sL = by_den(cmax), sR = by_den(cmin), sU = by_den(cmax * cmin);
    const double F = by_den(cmax * SL + cmin * SR - cmax * cmin * D);
    const double lcmax = by_den((SL - cmin * D) - F), lcmin = by_den((SR - cmax * D) - F);
    double lvxl = 0., lvxr = 0., lvnl = 0., lvnr = 0.;
    if (m1 > vxr) { if (!(0. > vxl)) lvxl = lcmax; }
    else lvxr = lcmax;
    if (n1 > -vnr) { if (!(0. > -vnl)) lvnl = -lcmin; }
    else lvnr = -lcmin;
    StateAdj a;
    contraction_vjp(pl, ql, cl, dir, gam, lf, sL, sU, a);
    vl.vjp(ql, dir, G, gam, lvxl, lvnl, a);
    state_pullback(pl, ql, G, L, a, lpl);
    contraction_vjp(pr, qr, cr, dir, gam, lf, sR, -sU, a);
    vr.vjp(qr, dir, G, gam, lvxr, lvnr, a);
    state_pullback(pr, qr, G, L, a, lpr);
}

}  // namespace hamr
