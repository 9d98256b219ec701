// gf_physics_fast.h -- the step's scalar routines for tiles whose cells,
// parameters and step sizes lie in the range of gf_exact.h: the same values as
// the general operations (gf_physics.h), except for the sign of a zero, with
// the quotients, roots, maxima and minima of gf_exact.h.  Terms that are exact
// zeros for finite values (Cramer's rule of the sparse eigenvector matrix, the
// second wave's two zero components) are left out, and lanes that take
// different cases form both and select, or multiply by 0 or 1: neither holds
// for an infinity or a NaN, which the range excludes.
//
// On the 4096^2 dam break a launch of the 32x32 step kernel (about 2,360 active
// patches) fell from 1.275e8 to 1.019e8 VALU instructions and from 346 to
// 284 us (with the other steps of the kernel since: 8.85e7 on 2,244 active
// patches, 250 us).
#pragma once

#include "gf_exact.h"
#include "gf_physics.h"

namespace gf {
namespace fast {

// Quotients of one cell's depth: for a wet cell hu/h, hv/h, sqrt(g h) and the
// reciprocal they share, formed once for the faces and splits that use them.
struct CellVel {
    double u, v, sg, y;
};

__device__ __forceinline__ CellVel cell_velocity(double h, double hu, double hv, double g)
{
    const Recip d = recip(h);
    return CellVel{quot(hu, d), quot(hv, d), root(g * h), d.y};
}

// Speeds s1m, s2m of riemanntype's middle state (geoclaw_riemann_utils.f:
// 566-677, maxiter = 1) for two depths above drytol.  rL, rR: the depths with
// their reciprocals; sgL, sgR = sqrt(g*hL), sqrt(g*hR): every sqrt(g*h) of hL,
// hR, h_min or h_max is one of them, bit for bit.
__device__ __forceinline__ void middle_speeds(const Recip& rL, const Recip& rR, double uL, double uR, double sgL,
                                              double sgR, const Params& P, double& s1m, double& s2m)
{
    const double hL = rL.b, hR = rR.b, g = P.grav, halfg = P.halfg;
    const bool left = !(hR > hL);  // the left depth is the larger, or they are equal
    const double h_min = left ? hR : hL;
    const double h_max = left ? hL : hR;
    const double dh = h_max - h_min;
    const double delu = uR - uL;
    const double F_min = delu + 2.0 * ((left ? sgR : sgL) - (left ? sgL : sgR));
    const double F_max = delu + dh * root(quot(halfg * (h_max + h_min), h_max * h_min));
    // two rarefactions and the shock-rarefaction pair are formed by every lane,
    // the two-shock case by the lanes that have it: a branch costs a wave more
    // than the few instructions of the first two
    const bool rare = F_min > 0.0, shocks = !rare && F_max <= 0.0;
    // F0 = delu + 2(sqrt(g h0) - sqrt(g h_max)) + (h0 - h_min) sqrt(g/2 (1/h0 + 1/h_min))
    // at h0 = h_min: the last product is zero
    const double F0 = F_min;
    const double tr = vmax(0.0, -delu + 2.0 * (sgL + sgR));
    double hm = rare ? P.inv16g * (tr * tr) : h_min - quot(F0, quot(F_max - F0, dh));
    double u1m = 0.0, u2m = 0.0;
    if (shocks) {
        // one Newton step on sqrt(h) from h0 = h_max.  The side at h0 has a zero
        // (h0 - h) factor: only the other side's terms remain, and 1/h0 is that
        // side's own 1/h
        const double i_max = quot(1.0, left ? rL : rR);
        const double i_min = quot(1.0, left ? rR : rL);
        const double gs = root(halfg * (i_max + i_max));
        const double go = root(halfg * (i_max + i_min));
        const double F0s = delu + dh * go;
        const double T = quot(g * dh, 4.0 * (h_max * h_max) * go);
        const double dfdh = left ? (gs + go) - T : (go - T) + gs;
        const double rh = root(h_max);
        const double slope = 2.0 * rh * dfdh;
        const double t = rh - quot(F0s, slope);
        hm = t * t;
        const double im = quot(1.0, hm);
        u1m = uL - (hm - hL) * root(halfg * (im + (left ? i_max : i_min)));
        u2m = uR + (hm - hR) * root(halfg * (im + (left ? i_min : i_max)));
    }
    const double sghm = root(g * hm);
    // two rarefactions:      s1m = (uL + 2 sqrt(g hL)) - 3 sghm, s2m = (uR - 2 sqrt(g hR)) + 3 sghm
    // shock-rarefaction:     hL > hR: a = uL + 2 sqrt(g hL), s1m = a - 3 sghm, s2m = a - sghm
    //                        else:    a = uR - 2 sqrt(g hR), s2m = a + 3 sghm, s1m = a + sghm
    // two shocks:            s1m = u1m - sghm, s2m = u2m + sghm
    const double A = uL + 2.0 * sgL, B = uR - 2.0 * sgR, s3 = 3.0 * sghm;
    const bool fromL = hL > hR;
    s1m = shocks ? u1m - sghm : (rare || fromL) ? A - s3 : B + sghm;
    s2m = shocks ? u2m + sghm : (rare || !fromL) ? B + s3 : A - sghm;
}

// hm of riemanntype(h, h, u, -u), h > drytol, the wall test of rpn2
// (rpn2_geoclaw.f:185-242), whose speeds the caller does not use.  With
// hL = hR = h every (h_max - h_min) factor is an exact +0: F_min = F_max =
// delu, a positive F takes the two-rarefaction branch and any other the
// two-shock branch with gL = gR and dfdh = gL + gL.
__device__ __forceinline__ double wall_hstar(const Recip& r, double u, double sg, const Params& P)
{
    const double delu = -u - u;
    if (delu > 0.0) {
        const double t = vmax(0.0, -delu + 2.0 * (sg + sg));
        return P.inv16g * (t * t);
    }
    const double ih = quot(1.0, r);
    const double gL = root(P.halfg * (ih + ih));
    const double rh = root(r.b);
    const double slope = 2.0 * rh * (gL + gL);
    const double t = rh - quot(delu, slope);
    return t * t;
}

// One face of rpn2 (rpn2_geoclaw.f:84-330) followed by riemann_aug_JCP
// (geoclaw_riemann_utils.f:2-311, maxiter = 1, no rarefaction corrector).
// Inputs are the left/right states in direction-local order (h, normal
// momentum, transverse momentum) and the left/right bathymetry.  Outputs: the
// speeds s[3] and the f-waves in compressed form, wave 1 (3), the normal
// momentum of wave 2, wave 3 (3): the other two components of wave 2 are exact
// zeros (geoclaw_riemann_utils.f:289-299: fw(1,2) = beta(2)*r(2,2) = 0,
// fw(3,2) = 0).  A face with both sides dry gives zeros, as the reference
// leaves them.  cL, cR: the two cells' velocities, sqrt(g h) and reciprocal
// depth, used where the cell is wet.
__device__ __forceinline__ void rpn2_face(double hL, double huL, double hvL, double bL,
                                          double hR, double huR, double hvR, double bR,
                                          const CellVel& cL, const CellVel& cR,
                                          const Params& P, double s[3], double w[7])
{
    const double g = P.grav, drytol = P.dry_tolerance, halfg = P.halfg;
    const bool wetL = hL > drytol, wetR = hR > drytol;
    const bool still = hL <= drytol && hR <= drytol;
    // Both sides as if wet; the lanes of a wave that have a dry side are put
    // right below, in code that the other waves skip.
    Recip rL{hL, cL.y}, rR{hR, cR.y};
    double uL = cL.u, vL = cL.v, sgL = cL.sg, uR = cR.u, vR = cR.v, sgR = cR.sg;
    double phiL = halfg * (hL * hL) + quot(huL * huL, rL);
    double phiR = halfg * (hR * hR) + quot(huR * huR, rR);
    const bool front = !(wetL && wetR);
    bool wallL = false, wallR = false;
    if (front) {
        if (!wetL) {
            hL = 0.0; huL = 0.0; hvL = 0.0; uL = 0.0; vL = 0.0; phiL = 0.0; sgL = 0.0;
        }
        if (!wetR) {
            hR = 0.0; huR = 0.0; hvR = 0.0; uR = 0.0; vR = 0.0; phiR = 0.0; sgR = 0.0;
        }
        // the wall test of whichever side is dry: riemanntype(hL, hL, uL, -uL) or
        // riemanntype(hR, hR, -uR, uR), one call for both kinds of lane; a dry
        // side that the water cannot climb is a wall (the wet side mirrored)
        const double hstar = wall_hstar(wetL ? rL : rR, wetL ? uL : -uR, wetL ? sgL : sgR, P);
        if (!wetR) {
            const double hstartest = fmaxf64(hL, hstar);
            if (hstartest + bL < bR) {
                wallR = true;
                hR = hL; huR = -huL; bR = bL; phiR = phiL; uR = -uL; vR = vL; sgR = sgL; rR = rL;
            } else if (hL + bL < bR) {
                bR = hL + bL;
            }
        } else {
            const double hstartest = fmaxf64(hR, hstar);
            if (hstartest + bR < bL) {
                wallL = true;
                hL = hR; huL = -huR; bL = bR; phiL = phiR; uL = -uR; vL = vR; sgL = sgR; rL = rR;
            } else if (hR + bR < bL) {
                bL = hR + bR;
            }
        }
    }

    const double sL = uL - sgL;
    const double sR = uR + sgR;
    const double uhat = quot(sgL * uL + sgR * uR, sgR + sgL);
    const double chat = root(halfg * (hR + hL));
    const double sRoe1 = uhat - chat;
    const double sRoe2 = uhat + chat;

    // ---- riemann_aug_JCP ----
    const double delh = hR - hL;
    const double delhu = huR - huL;
    const double delphi = phiR - phiL;
    const double delb = bR - bL;

    double s1m, s2m;
    middle_speeds(rL, rR, uL, uR, sgL, sgR, P, s1m, s2m);
    if (front && fminf64(hR, hL) <= drytol) {
        s1m = uR + uL - 2.0 * sgR + 2.0 * sgL;
        s2m = s1m;
    }

    // (the sign of a zero speed matters to the limiter; in the fast range these
    // are sums, whose zeros are all +0)
    const double sE1 = vmin(vmin(sL, sRoe1), s2m);
    const double sE2 = vmax(vmax(sR, sRoe2), s1m);
    const double lam0 = sE1, lam2 = sE2;
    const double lam1 = 0.5 * (lam0 + lam2);
    // r(:,1) = (1, lam0, lam0^2), r(:,2) = (0, 0, 1), r(:,3) = (1, lam2, lam2^2)
    const double r10 = lam0, r20 = lam0 * lam0;
    const double r12 = lam2, r22 = lam2 * lam2;

    // a level bed has delb = 0, and with it deldelh = deldelphi = 0 whatever
    // the bounds below (each lies on the other side of 0)
    double deldelh = 0.0, deldelphi = 0.0;
    if (delb != 0.0) {
        const double hstarHLL = vmax(quot(huL - huR + sE2 * hR - sE1 * hL, sE2 - sE1), 0.0);
        const double crit = P.crit, crit2 = P.crit2;
        const double hbar = vmax(0.5 * (hL + hR), 0.0);
        const double tu = uL + uR;
        const double s1s2bar = 0.25 * (tu * tu) - g * hbar;
        const double s1s2tilde = vmax(0.0, uL * uR) - g * hbar;
        const bool sonic = (fabs(s1s2bar) <= crit) | (s1s2bar * s1s2tilde <= P.critsq) |
                           (s1s2bar * sE1 * sE2 <= P.critsq) | (vmin(fabs(sE1), fabs(sE2)) < crit2) |
                           ((sE1 < crit2) & (s1m > -crit2)) | ((sE2 > -crit2) & (s2m < crit2)) |
                           ((uL + sgL) * (uR + sgR) < 0.0) | ((uL - sgL) * (uR - sgR) < 0.0);
        const Recip rb = recip(s1s2bar);
        const double gb = delb * g * hbar, gn = -delb * g * hbar;
        deldelh = sonic ? -delb : quot(gb, rb);
        // the bounds' two quotients are formed once for every lane (the three
        // cases use them in different combinations)
        const double hs = hstarHLL * (sE2 - sE1);
        const double q2 = quot(hs, sE2);
        const double q1 = quot(hs, sE1);
        const bool sub = sE1 < -crit && sE2 > crit, right = !sub && sE1 >= crit, left = !sub && !right && sE2 <= -crit;
        const double upper = sub ? q2 : right ? q1 : hR, lower = sub ? q1 : right ? -hL : q2;
        const double bounded = vmax(vmin(deldelh, upper), lower);
        deldelh = (sub || right || left) ? bounded : deldelh;
        deldelphi = sonic ? -g * hbar * delb : quot(gn * s1s2tilde, rb);
        deldelphi = vmin(deldelphi, g * vmax(-hL * delb, -hR * delb));
        deldelphi = vmax(deldelphi, g * vmin(-hL * delb, -hR * delb));
    }

    const double d0 = delh - deldelh;
    const double d1 = delhu;
    const double d2 = delphi - deldelphi;

    // Cramer's rule as the reference writes it (geoclaw_riemann_utils.f:230-249)
    // with r = [[1,0,1],[r10,0,r12],[r20,1,r22]], its zero terms left out
    const Recip det = recip(r10 - r12);
    const double beta0 = quot(d1 - d0 * r12, det);
    const double beta1 = quot(((d1 * r22 - r12 * d2) - d0 * (r10 * r22 - r12 * r20)) + (r10 * d2 - d1 * r20), det);
    const double beta2 = quot(d0 * r10 - d1, det);

    // f-waves (geoclaw_riemann_utils.f:289-306)
    const double fw00 = beta0 * r10, fw20 = beta2 * r12;
    double fw02 = fw00 * vL, fw22 = fw20 * vR;
    const double rest = hR * uR * vR - hL * uL * vL - fw02 - fw22;
    const bool below = huL + fw00 <= 0.0;
    fw02 = below ? fw02 + rest : fw02;
    fw22 = below ? fw22 : fw22 + rest;

    s[0] = lam0; s[1] = lam1; s[2] = lam2;
    w[0] = fw00; w[1] = beta0 * r20; w[2] = fw02;
    w[3] = beta1;
    w[4] = fw20; w[5] = beta2 * r22; w[6] = fw22;
    if (front) {
        // eliminate ghost fluxes for the wall problem (rpn2_geoclaw.f:303-309);
        // no waves between dry cells (there the products are of garbage)
        const double w0 = wallL ? 0.0 : 1.0, w1 = wallL || wallR ? 0.0 : 1.0, w2 = wallR ? 0.0 : 1.0;
        const double f[3] = {w0, w1, w2};
#pragma unroll
        for (int k = 0; k < 3; k++) s[k] = still ? 0.0 : s[k] * f[k];
#pragma unroll
        for (int k = 0; k < 7; k++) w[k] = still ? 0.0 : w[k] * f[k / 3 < 1 ? 0 : (k == 3 ? 1 : 2)];
    }
}

// Fluctuations of one face (rpn2_geoclaw.f:359-376) from its compressed
// waves, direction-local order: a wave goes to amdq when its speed is
// negative, to apdq when it is positive and half to each at zero, i.e. times
// 1, 1/2 or 0 to each (exact products).
__device__ __forceinline__ void fluctuations(const double s[3], const double w[7], double amdq[3], double apdq[3])
{
    double cm[3], cp[3];
#pragma unroll
    for (int mw = 0; mw < 3; mw++) {
        cm[mw] = s[mw] < 0.0 ? 1.0 : (s[mw] > 0.0 ? 0.0 : 0.5);
        cp[mw] = 1.0 - cm[mw];
    }
    amdq[0] = cm[0] * w[0] + cm[2] * w[4];
    amdq[1] = cm[0] * w[1] + cm[1] * w[3] + cm[2] * w[5];
    amdq[2] = cm[0] * w[2] + cm[2] * w[6];
    apdq[0] = cp[0] * w[0] + cp[2] * w[4];
    apdq[1] = cp[0] * w[1] + cp[1] * w[3] + cp[2] * w[5];
    apdq[2] = cp[0] * w[2] + cp[2] * w[6];
}

// The limiter function of philim (philim.f:65-126) at the ratio r = b / a,
// a != 0; an out-of-range method falls through to minmod.
__device__ __forceinline__ double philim(double r, int meth)
{
    switch (meth) {
    case 2:
        return vmax(vmax(0.0, vmin(1.0, 2.0 * r)), vmin(2.0, r));
    case 3:
        return (r + fabs(r)) / (1.0 + fabs(r));
    case 4: {
        const double c = (1.0 + r) / 2.0;
        return vmax(0.0, vmin(vmin(c, 2.0), 2.0 * r));
    }
    case 5:
        return r;
    default:
        return vmax(0.0, vmin(1.0, r));
    }
}

// Some non-zero value of the N is too small for quot as a numerator or
// denominator (gf_exact.h).
template <int N>
__device__ __forceinline__ bool quotients_tiny(const double (&a)[N])
{
    int e = 0;
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int x = exponent_of(a[k]);
        e = x < e ? x : e;
    }
    return e < QUOT_MIN_EXP;
}

// Eigen-split of a transverse fluctuation for one cell (rpt2_geoclaw.f:61-187):
// the cell's velocities (u normal, v transverse with respect to the normal
// solve), its surface eta = h + b and the bathymetry of its two transverse
// neighbours.  The split is applied to two fluctuations (the imp = 1 split of
// amdq of the face on the cell's right/top and the imp = 2 split of apdq of
// the face on its left/bottom share the same Jacobian).
struct Rpt2Cell {
    bool active, lo, hi;  // lo / hi: the surface reaches the neighbour below / above
    double u, s0, s1, s2;
};

__device__ __forceinline__ Rpt2Cell rpt2_setup(double h, double u, double v, double sg, double b,
                                               double topo1, double topo3, double tol)
{
    Rpt2Cell c;
    const double eta = h + b;
    c.active = !(h <= tol) && !(eta < vmin(topo1, topo3));
    c.lo = eta >= topo1;
    c.hi = eta >= topo3;
    c.u = u;
    c.s0 = v - sg;
    c.s1 = v;
    c.s2 = v + sg;
    return c;
}

// One side's sum over the waves of speed * beta * r with r(:,1) = (1, u, s0),
// r(:,2) = (0, 1, 0), r(:,3) = (1, u, s2); sp is 0 for a wave that does not
// go there.
__device__ __forceinline__ void rpt2_side(const double sp[3], const double beta[3], const Rpt2Cell& c, double out[3])
{
    const double t0 = sp[0] * beta[0], t1 = sp[1] * beta[1], t2 = sp[2] * beta[2];
    out[0] = t0 + t2;
    out[1] = t0 * c.u + t1 + t2 * c.u;
    out[2] = t0 * c.s0 + t2 * c.s2;
}

// Transverse increments of one cell from the two normal fluctuations that its
// state splits (geoclaw_flux2fw_fort.f:232-265): G1 (below/left) and G2
// (above/right), direction-local order, hd = dt/dx / 2.
__device__ __forceinline__ void cell_transverse(const Rpt2Cell& c, const double am_next[3], const double ap_own[3],
                                                double hd, double G1[3], double G2[3])
{
#pragma unroll
    for (int k = 0; k < 3; k++) { G1[k] = 0.0; G2[k] = 0.0; }
    if (!c.active) return;
    const double den = c.s2 - c.s0;
    const double n[4] = {c.s2 * am_next[0] - am_next[2], am_next[2] - c.s0 * am_next[0],
                         c.s2 * ap_own[0] - ap_own[2], ap_own[2] - c.s0 * ap_own[0]};
    double be[4];
    const Recip r = recip(den);
#pragma unroll
    for (int k = 0; k < 4; k++) be[k] = quot(n[k], r);
    if (quotients_tiny(n)) {
#pragma unroll
        for (int k = 0; k < 4; k++) be[k] = n[k] / den;
    }
    const double b1[3] = {be[0], -c.u * am_next[0] + am_next[1], be[1]};
    const double b2[3] = {be[2], -c.u * ap_own[0] + ap_own[1], be[3]};
    // the waves that go down are those of negative speed, where the surface
    // reaches the bed below, and the others count with speed 0; likewise up
    const double dn[3] = {vmin(c.s0, 0.0), vmin(c.s1, 0.0), vmin(c.s2, 0.0)};
    const double up[3] = {vmax(c.s0, 0.0), vmax(c.s1, 0.0), vmax(c.s2, 0.0)};
    const double hlo = c.lo ? hd : 0.0, hhi = c.hi ? hd : 0.0;
    double d1[3], d2[3];
    rpt2_side(dn, b1, c, d1);
    rpt2_side(dn, b2, c, d2);
#pragma unroll
    for (int k = 0; k < 3; k++) G1[k] = -(hlo * d1[k]) - hlo * d2[k];
    rpt2_side(up, b1, c, d1);
    rpt2_side(up, b2, c, d2);
#pragma unroll
    for (int k = 0; k < 3; k++) G2[k] = -(hhi * d1[k]) - hhi * d2[k];
}

// Manning friction of fc2d_geoclaw_src2 (geoclaw_src2_fort.f90:41-71) for one
// interior cell; manning_break(1) = rinfinity (default-real 10.e32).
__device__ __forceinline__ void src2_cell(double h, double& hu, double& hv, double b,
                                          double dt, const Params& P)
{
    if (!P.friction_forcing) return;
    if (h < 1.0e-30) {
        hu = 0.0;
        hv = 0.0;
    } else if (h <= P.friction_depth) {
        const double coeff = (b < (double)10.e32f) ? P.manning_n : 0.0;
        const double c2 = coeff * coeff;
        const double sq = hu * hu + hv * hv;
        const double pw = pow_7_3(h);
        // momenta above 2^-300 and a friction term of ordinary size, or none
        const double num = root(sq) * P.grav * c2;
        const double lo = vmin(hu == 0.0 ? 1.0 : fabs(hu), hv == 0.0 ? 1.0 : fabs(hv));
        const Recip d = recip(1.0 + dt * quot(num, pw));
        if (sq < 0x1p600 && lo >= 0x1p-300 && (num >= 0x1p-400 || num == 0.0) && d.b < 0x1p300) {
            hu = quot(hu, d);
            hv = quot(hv, d);
        } else {
            const double gamma = sqrt(sq) * P.grav * c2 / pw;
            const double dgamma = 1.0 + dt * gamma;
            hu = hu / dgamma;
            hv = hv / dgamma;
        }
    }
}

// Limiter, second-order correction and fluctuation split of one face
// (geoclaw_flux2fw_fort.f:143-224 with geoclaw_limiter_fort.f:34-58 and
// philim.f).  w: own compressed unlimited waves; wn: for each wave that of the
// face it comes from (load_waves).  Outputs in direction-local order: faddm,
// faddp (flux increments) and amdq*, apdq* (fluctuations handed to rpt2).
// DEF: the default method (order 2, transverse 2, MC limiter on all three
// families) fixed at compile time; otherwise the method is read from P.
template <int DIR, bool DEF>
__device__ __forceinline__ void face_second_order(const double w[7], const double s[3],
                                                  const double wn[7], double dtdx, const Params& P,
                                                  double faddm[3], double faddp[3],
                                                  double amq[3], double apq[3])
{
    double amdq[3], apdq[3];
    fluctuations(s, w, amdq, apdq);
    const int order = DEF ? 2 : P.order;
    if (order == 1) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            faddm[k] = amdq[k];
            faddp[k] = -apdq[k];
            amq[k] = amdq[k];
            apq[k] = apdq[k];
        }
        return;
    }
    // limiter on the three wave families (wave 2 has its normal momentum only):
    // the ratios b / a of the dot products, then the factor of each family (1
    // where the wave vanishes or its family is not limited)
    const double a[3] = {pdot<DIR>(w, w), w[3] * w[3], pdot<DIR>(w + 4, w + 4)};
    const double b[3] = {pdot<DIR>(wn, w), wn[3] * w[3], pdot<DIR>(wn + 4, w + 4)};
    double r[3];
#pragma unroll
    for (int mw = 0; mw < 3; mw++) r[mw] = quot(b[mw], a[mw]);
    const double ab[6] = {a[0], a[1], a[2], b[0], b[1], b[2]};
    if (quotients_tiny(ab)) {
#pragma unroll
        for (int mw = 0; mw < 3; mw++) r[mw] = b[mw] / a[mw];
    }
    double lim[3], c[3];
#pragma unroll
    for (int mw = 0; mw < 3; mw++) {
        const int meth = DEF ? 4 : P.mthlim[mw];
        lim[mw] = a[mw] != 0.0 && (DEF || meth != 0) ? philim(r[mw], meth) : 1.0;
        c[mw] = copysign(1.0, s[mw]) * (1.0 - fabs(s[mw]) * dtdx);
    }
    double cq[3];
    cq[0] = c[0] * (lim[0] * w[0]) + c[2] * (lim[2] * w[4]);
    cq[1] = c[0] * (lim[0] * w[1]) + c[1] * (lim[1] * w[3]) + c[2] * (lim[2] * w[5]);
    cq[2] = c[0] * (lim[0] * w[2]) + c[2] * (lim[2] * w[6]);
    const bool fold = DEF ? true : (P.transverse == 2);
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const double hq = 0.5 * cq[k];
        faddm[k] = amdq[k] + hq;
        faddp[k] = -apdq[k] + hq;
        amq[k] = fold ? amdq[k] + cq[k] : amdq[k];
        apq[k] = fold ? apdq[k] - cq[k] : apdq[k];
    }
}

}  // namespace fast
}  // namespace gf
