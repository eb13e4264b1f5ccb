// hc_fused_flux.hpp -- FP64 face arithmetic of the fused Euler kernels: limiters and flux functors in
// the form with the fewest operations, for the same schemes as hc_point.hpp (which keeps the
// reference's operation order and is what these are tested against).
//
// What changes against hc_point.hpp, and why the results agree to rounding:
//  - one reciprocal per state (1/rho) instead of a division per quantity; p / (rho R) and the factors
//    of R around it cancel: a^2 = gamma p / rho, h = a^2/(gamma-1) + k;
//  - square roots and reciprocals of hc_arith.hpp, and the reciprocal sound speed from the root's seed;
//  - products and sums fused (explicit fma, so every kernel that uses a function rounds alike);
//  - face-frame Roe: the jumps of the primitive variables enter the characteristic waves directly.  For
//    Roe's average, d(rho u) = rho~ du + u~ drho and d(rho E) = dp/(gamma-1) + rho~ u~.du + k~ drho
//    hold exactly, so the transformation of the conserved jump to primitive variables and the four
//    basis changes collapse (390 -> 190 instructions per face with the central flux);
//  - AUSM+up: the supersonic pressure splitting of machSplittings.ipp:27-34 is
//    (m1 + eps) / (|M| + eps) with eps the largest number, which is 1 for every |M| below 2^970.
#pragma once

#include "hc_point.hpp"

namespace hc {

// the state quantities the flux functors read
struct FState {
    double r, u, v, p, h, a2;
};

template <int BASIS> HC_HD FState fused_state(const Species<double>& sp, const double* q)
{
    FState s;
    if constexpr (BASIS == BASIS_PRIMITIVE) {
        s.u = q[0];
        s.v = q[1];
        s.r = q[2];
        s.p = q[3];
        const double k = 0.5 * hc_fma(s.u, s.u, s.v * s.v);
        s.a2 = sp.gamma * s.p * hc_rcp(s.r);
        s.h = hc_fma(s.a2, sp.gamma1, k);
    } else {
        s.r = q[2];
        const double ri = hc_rcp(s.r);
        s.u = q[0] * ri;
        s.v = q[1] * ri;
        const double rk = 0.5 * hc_fma(q[0], s.u, q[1] * s.v);
        s.p = (sp.gamma - 1.0) * (q[3] - rk);
        s.a2 = sp.gamma * s.p * ri;
        s.h = (q[3] + s.p) * ri;
    }
    return s;
}

// conserved variables of a state
HC_HD void fused_conserved(const FState& s, double* c)
{
    c[0] = s.r * s.u;
    c[1] = s.r * s.v;
    c[2] = s.r;
    c[3] = hc_fma(s.r, s.h, -s.p);
}

// sum of the two states' exact fluxes (euler/fluxes/exactFlux.ipp:4-36)
HC_HD void fused_exact_sum(double n0, double n1, const FState& L, const FState& R, double unl, double unr, double* f)
{
    const double ml = L.r * unl, mr = R.r * unr, ps = L.p + R.p;
    f[0] = hc_fma(mr, R.u, hc_fma(ml, L.u, ps * n0));
    f[1] = hc_fma(mr, R.v, hc_fma(ml, L.v, ps * n1));
    f[2] = ml + mr;
    f[3] = hc_fma(mr, R.h, ml * L.h);
}

// |l| with Harten's fix (euler/fluxes/roe.ipp:50-78): l, ll, lr the wave's speed in the average and
// in the left and right states
HC_HD double fused_harten(double l, double ll, double lr)
{
    const double e = 0.05 * hc_fmax(0.0, hc_fmax(l - ll, lr - l));
    const double a = hc_fabs(l);
    return a >= e ? a : 0.5 * (e + a * a * hc_rcp(e));
}

// Roe average (euler/fluxes/roe.ipp:2-48) with its sound speed and the reciprocal of it
struct FRoe {
    double r, u, v, h, k, a, ai, un;
};
HC_HD FRoe fused_roe_average(const Species<double>& sp, double n0, double n1, const FState& L, const FState& R, double du,
                             double dv)
{
    FRoe w;
    const double cr = hc_root(R.r * hc_rcp(L.r));
    const double wl = hc_rcp(1.0 + cr);
    w.r = cr * L.r;
    w.u = hc_fma(-wl, du, R.u);
    w.v = hc_fma(-wl, dv, R.v);
    w.h = hc_fma(wl, L.h - R.h, R.h);
    w.k = 0.5 * hc_fma(w.u, w.u, w.v * w.v);
    w.a = hc_root((sp.gamma - 1.0) * (w.h - w.k), w.ai);
    w.un = hc_fma(n0, w.u, n1 * w.v);
    return w;
}

// Roe (base/fluxes/roeFlux.ipp:2-58) with the averaged velocity in the face frame: the waves of the
// velocity and pressure jumps, scaled, as momentum, density and energy
HC_HD void fused_roe(const Species<double>& sp, double area, double n0, double n1, const FState& L, const FState& R, double* F,
                     double& lam)
{
    const double unl = hc_fma(n0, L.u, n1 * L.v), unr = hc_fma(n0, R.u, n1 * R.v);
    const double al = hc_root(L.a2), ar = hc_root(R.a2);
    const double du = R.u - L.u, dv = R.v - L.v;
    const FRoe w = fused_roe_average(sp, n0, n1, L, R, du, dv);
    const double s0 = hc_fabs(w.un);
    const double s1 = fused_harten(w.un - w.a, unl - al, unr - ar);
    const double s2 = fused_harten(w.un + w.a, unl + al, unr + ar);
    const double rdn = w.r * hc_fma(n0, du, n1 * dv), dpa = (R.p - L.p) * w.ai;
    const double m1 = s1 * (rdn - dpa), m2 = s2 * (rdn + dpa);          // the acoustic waves
    const double md = 0.5 * (m2 - m1);
    const double wn = 0.5 * (m1 + m2);                                  // rho du_n
    const double wt = s0 * (w.r * hc_fma(n0, dv, -(n1 * du)));          // rho du_t
    const double wr = hc_fma(md, w.ai, s0 * hc_fma(-dpa, w.ai, R.r - L.r));   // drho
    const double ut = hc_fma(n0, w.v, -(n1 * w.u));
    double f[4];
    fused_exact_sum(n0, n1, L, R, unl, unr, f);
    f[0] = f[0] - hc_fma(n0, wn, hc_fma(-n1, wt, w.u * wr));
    f[1] = f[1] - hc_fma(n1, wn, hc_fma(n0, wt, w.v * wr));
    f[2] = f[2] - wr;
    f[3] = f[3] - hc_fma(md * w.a, sp.gamma1, hc_fma(w.un, wn, hc_fma(ut, wt, w.k * wr)));
    const double c = 0.5 * area;
    for (int v = 0; v < 4; ++v) F[v] = f[v] * c;
    lam = hc_fmax(s0 + w.a, hc_fmax(hc_fabs(unl) + al, hc_fabs(unr) + ar)) * area;
}

// RoeUnprecWS (euler/fluxes/roeUnprecWS.ipp:24-104; coefficients as in hc_point.hpp)
HC_HD void fused_roe_unprec_ws(const Species<double>& sp, double area, double n0, double n1, const FState& L,
                               const FState& R, double* F, double& lam)
{
    const double unl = hc_fma(n0, L.u, n1 * L.v), unr = hc_fma(n0, R.u, n1 * R.v);
    const double al = hc_root(L.a2), ar = hc_root(R.a2);
    const double dp = R.p - L.p, du = unr - unl;
    const FRoe w = fused_roe_average(sp, n0, n1, L, R, R.u - L.u, R.v - L.v);
    const double minf = sp.minf, uinf = minf * w.a;
    const double dU = hc_fma(minf * hc_rcp(w.r * uinf * uinf), dp, 0.05 * du);
    const double dP = hc_fma(0.02 * minf, dp, 0.10 * (w.r * uinf) * minf * du);
    const double s0 = hc_fabs(w.un), rU = w.r * dU;
    double cl[4], cr[4], f[4];
    fused_conserved(L, cl);
    fused_conserved(R, cr);
    fused_exact_sum(n0, n1, L, R, unl, unr, f);
    f[0] = f[0] - hc_fma(s0, cr[0] - cl[0], hc_fma(rU, w.u, dP * n0));
    f[1] = f[1] - hc_fma(s0, cr[1] - cl[1], hc_fma(rU, w.v, dP * n1));
    f[2] = f[2] - hc_fma(s0, cr[2] - cl[2], rU);
    f[3] = f[3] - hc_fma(s0, cr[3] - cl[3], hc_fma(rU, w.h, dP * w.un));
    const double c = 0.5 * area;
    for (int v = 0; v < 4; ++v) F[v] = f[v] * c;
    lam = hc_fmax(s0 + w.a, hc_fmax(hc_fabs(unl) + al, hc_fabs(unr) + ar)) * area;
}

// central and Rusanov (base/fluxes/centralFlux.ipp:2-14, rusanovFlux.ipp:2-50)
template <bool RUSANOV>
HC_HD void fused_central(double area, double n0, double n1, const FState& L, const FState& R, double* F, double& lam)
{
    const double unl = hc_fma(n0, L.u, n1 * L.v), unr = hc_fma(n0, R.u, n1 * R.v);
    const double s = hc_fmax(hc_fabs(unl) + hc_root(L.a2), hc_fabs(unr) + hc_root(R.a2));
    double f[4];
    fused_exact_sum(n0, n1, L, R, unl, unr, f);
    if constexpr (RUSANOV) {
        double cl[4], cr[4];
        fused_conserved(L, cl);
        fused_conserved(R, cr);
        for (int v = 0; v < 4; ++v) f[v] = hc_fma(-s, cr[v] - cl[v], f[v]);
    }
    const double c = 0.5 * area;
    for (int v = 0; v < 4; ++v) F[v] = f[v] * c;
    lam = s * area;
}

// mass flux times the upwind side's (u, v, 1, h), plus the pressure (ausmPlusUP.ipp:155-171)
HC_HD void fused_convect(double mdot, bool left, double p, double n0, double n1, const FState& L, const FState& R, double* F)
{
    F[0] = hc_fma(mdot, left ? L.u : R.u, p * n0);
    F[1] = hc_fma(mdot, left ? L.v : R.v, p * n1);
    F[2] = mdot;
    F[3] = mdot * (left ? L.h : R.h);
}

// AUSM+up (euler/fluxes/ausmPlusUP.ipp:6-171): alpha0 = 3/16, beta = 1/8, Ku = 1.5, Kp = 0.25, sigma = 1
HC_HD void fused_ausmpup(const Species<double>& sp, int vscale, int pscale, double area, double n0, double n1, bool wl,
                         const FState& L, const FState& R, double* F, double& lam)
{
    const double asc = 2.0 * (sp.gamma - 1.0) * hc_rcp(sp.gamma + 1.0);
    const double unl = hc_fma(n0, L.u, n1 * L.v), unr = hc_fma(n0, R.u, n1 * R.v);
    const double als2 = asc * L.h, ars2 = asc * R.h;
    const double als = als2 * hc_rcp(hc_fmax(unl, hc_root(als2)));
    const double ars = ars2 * hc_rcp(hc_fmax(-unr, hc_root(ars2)));
    const double as = hc_fmin(ars, als), asi = hc_rcp(as);
    const double ra = 0.5 * (L.r + R.r);
    const double ml = unl * asi, mr = unr * asi;
    const double m02 = 0.5 * hc_fma(ml, ml, mr * mr);
    const double m0 = hc_root(m02);
    const double m0c = std_clamp(m0, sp.minf, 1.0);
    double m0a = m0c;
    if (pscale == SCALE_ADAPTIVE || vscale == SCALE_ADAPTIVE)   // the species' dt may be infinite: IEEE division
        m0a = std_clamp(hc_fmax(m0, sp.lref / (as * sp.dt)), sp.minf, 1.0);
    const double m0p = pscale == SCALE_CONVECTIVE ? m0c : pscale == SCALE_ACOUSTIC ? 1.0 : m0a;
    const double m0u = vscale == SCALE_CONVECTIVE ? m0c : vscale == SCALE_ACOUSTIC ? 1.0 : m0a;
    const double fap = m0p * (2.0 - m0p), fau = m0u * (2.0 - m0u);
    const double frr = hc_rcp(fap * ra);                        // 1 / (fa_p rho)
    // the splittings' quadratic pieces m2(+-) of either side
    const double lp = 0.25 * (ml + 1.0) * (ml + 1.0), lm = -0.25 * (ml - 1.0) * (ml - 1.0);
    const double rp = 0.25 * (mr + 1.0) * (mr + 1.0), rm = -0.25 * (mr - 1.0) * (mr - 1.0);
    const bool supl = hc_fabs(ml) > 1.0, supr = hc_fabs(mr) > 1.0;
    const double mlp = supl ? hc_fmax(ml, 0.0) : hc_fma(-2.0 * lp, lm, lp);
    const double mrm = supr ? hc_fmin(mr, 0.0) : hc_fma(2.0 * rm, rp, rm);
    const double dp = R.p - L.p;
    const double mp = 0.25 * hc_fmax(1.0 - m02, 0.0) * dp * (frr * asi * asi);
    const double ua = as * (mlp + mrm - mp) * area;
    const double al16 = 3.0 * hc_fma(5.0 * fau, fau, -4.0);     // 16 alpha
    const double plp = supl ? 1.0 : lp * hc_fma(-al16 * ml, lm, 2.0 - ml);
    const double prm = supr ? 1.0 : rm * hc_fma(al16 * mr, rp, -2.0 - mr);
    const double pu = 1.5 * plp * prm * ra * (fau * as) * (unr - unl);
    const double pa = (hc_fma(plp, L.p, prm * R.p) - pu) * area;
    const bool left = ua > 0.0;
    fused_convect(ua * (left ? L.r : R.r), left, pa, n0, n1, L, R, F);
    lam = 0.0;
    if (!wl) return;   // wave-uniform
    const double lmd = 0.5 * (m0p + 1.0) * (frr * ra);
    const double amax = hc_root(hc_fmax(as * as, hc_fmax(L.a2, R.a2)));
    lam = hc_fma(lmd, amax, hc_fmax(hc_fabs(ua), hc_fmax(hc_fabs(unl), hc_fabs(unr)))) * area;
}

// FluxInterface (base/base.h:370-397) on face states in the solution basis; wl: lam is wanted
template <int BASIS, int FLUX>
HC_HD void fused_flux(const Species<double>& sp, int vscale, int pscale, double area, double n0, double n1, bool wl,
                      const double* ql, const double* qr, double* F, double& lam)
{
    const FState L = fused_state<BASIS>(sp, ql);
    const FState R = fused_state<BASIS>(sp, qr);
    if constexpr (FLUX == FLUX_CENTRAL) fused_central<false>(area, n0, n1, L, R, F, lam);
    else if constexpr (FLUX == FLUX_RUSANOV) fused_central<true>(area, n0, n1, L, R, F, lam);
    else if constexpr (FLUX == FLUX_ROE_FACEFRAME) fused_roe(sp, area, n0, n1, L, R, F, lam);
    else if constexpr (FLUX == FLUX_ROE_UNPREC_WS) fused_roe_unprec_ws(sp, area, n0, n1, L, R, F, lam);
    else fused_ausmpup(sp, vscale, pscale, area, n0, n1, wl, L, R, F, lam);
}

// Limiter L of a centred increment a with a biased one b (limiters/limiter.ipp).  van Albada:
// b a^2 + a b^2 = ab (a + b), and the switch on a b < 0 is a maximum with zero; MinMod: the part of the
// biased increment that has the sign of a, up to |a| (a NaN increment, beside a NaN state, has none
// and gives 0 like limit_fn).
template <int L> HC_HD double fused_limit(double a, double b)
{
    if constexpr (L == LIM_VANALBADA2 || L == LIM_SMOOTHVANALBADA) {
        double p = a * b;
        if constexpr (L == LIM_VANALBADA2) p = hc_fmax(p, 0.0);
        return p * (a + b) * hc_rcp(hc_fma(b, b, hc_fma(a, a, DBL_MIN)));
    } else if constexpr (L == LIM_MINMOD2) {
        const double sgn = hc_copysign(1.0, a);
        return hc_copysign(hc_fmin(hc_fmax(b * sgn, 0.0), hc_fabs(a)), a);
    } else {
        return limit_fn<L>(a, b);
    }
}

// one branch on the limiter's id per face, straight-line code over the variables
HC_HD void fused_limit4(int lim, const double* al, const double* bl, const double* ar, const double* br, double* sl, double* sr)
{
    switch (lim) {
#define HC_LIM_CASE(L)                              \
    case L:                                         \
        for (int v = 0; v < 4; ++v) {               \
            sl[v] = fused_limit<L>(al[v], bl[v]);   \
            sr[v] = fused_limit<L>(ar[v], br[v]);   \
        }                                           \
        return;
        HC_FOR_EACH_LIMITER(HC_LIM_CASE)
#undef HC_LIM_CASE
    default:
        for (int v = 0; v < 4; ++v) {
            sl[v] = fused_limit<LIM_SMOOTHVANALBADA>(al[v], bl[v]);
            sr[v] = fused_limit<LIM_SMOOTHVANALBADA>(ar[v], br[v]);
        }
    }
}

}   // namespace hc
