"""Host build of the step's scalar routines (geoflood_amd/csrc/gf_physics.h,
the general operations, and gf_physics_fast.h, those of tiles inside the range
of gf_exact.h; the same sources the device compiles) as one patch step in the
order of the step kernel.  The seeds of the reciprocal and the reciprocal
square root are the host's quotients cut to 25 bits: the refinement has to
bring them, as the device's, to the same values."""
import ctypes as ct
import os
import subprocess
import tempfile

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_LIB = None

_SRC = r'''
#include <cmath>
#include <cstring>
#include <vector>
#define __device__
#define __forceinline__ inline
#define GF_DEVICE inline
#define GF_HOST_DEVICE
#define GF_SEED_FUNCTIONS
namespace gf {
inline double cut(double x)
{
    unsigned long long b;
    std::memcpy(&b, &x, 8);
    b &= ~((1ull << 28) - 1);
    std::memcpy(&x, &b, 8);
    return x;
}
inline double rcp_seed(double b) { return cut(1.0 / b); }
inline double rsq_seed(double b) { return cut(1.0 / std::sqrt(b)); }
inline int exponent_of(double a)
{
    int e = 0;
    if (std::isfinite(a)) (void)std::frexp(a, &e);
    return e;
}
}
#include "gf_physics_fast.h"

namespace gf {
struct HostParams {
    double grav, dry_tolerance, manning_n, friction_depth;
    int friction_forcing, src_term, order, transverse, mthlim[3];
};

static Params params(const HostParams& h)
{
    Params P{};
    P.grav = h.grav;
    P.dry_tolerance = h.dry_tolerance;
    P.manning_n = h.manning_n;
    P.friction_depth = h.friction_depth;
    P.friction_forcing = h.friction_forcing;
    P.src_term = h.src_term;
    P.order = h.order;
    P.transverse = h.transverse;
    for (int k = 0; k < 3; k++) P.mthlim[k] = h.mthlim[k];
    P.halfg = 0.5 * P.grav;
    const double c = P.dry_tolerance * P.grav;
    P.crit = c > 1e-6 ? c : 1e-6;
    P.crit2 = std::sqrt(P.crit);
    P.critsq = P.crit * P.crit;
    P.inv16g = 1.0 / (16.0 * P.grav);
    P.fast = step_params_in_range(P.grav, P.dry_tolerance);
    return P;
}

// q: [ny+4][nx+4][3], b: [ny+4][nx+4], interior of q updated in place.
// Returns the largest CFL number, uncapped; in_range: the tile test.
extern "C" double gf_host_step(int fast_form, int nx, int ny, double* q, const double* bed, double dx, double dy, double dt,
                               const HostParams* hp, int* in_range)
{
    const Params P = params(*hp);
    const int W = nx + 4, NC = W * (ny + 4), PX = nx + 3, PY = ny + 3;
    const auto ti = [&](int i, int j) { return (j + 1) * W + i + 1; };
    const auto at = [&](int i, int j) { return j * PX + i; };
    const double dtdx = dt / dx, dtdy = dt / dy, tol = P.dry_tolerance, g = P.grav;
    std::vector<double> h(NC), hu(NC), hv(NC);
    bool ok = P.fast && dtdx >= 0x1p-100 && dtdx <= 0x1p100 && dtdy >= 0x1p-100 && dtdy <= 0x1p100, wet = false;
    for (int c = 0; c < NC; c++) {
        h[c] = q[3 * c];
        hu[c] = q[3 * c + 1];
        hv[c] = q[3 * c + 2];
        if (h[c] < tol) {
            h[c] = fmaxf64(h[c], 0.0);
            hu[c] = hv[c] = 0.0;
        }
        wet |= h[c] > tol;
        ok &= step_cell_in_range(h[c], hu[c], hv[c], bed[c]);
    }
    *in_range = ok;
    struct V3 { double v[3]; };
    struct V7 { double v[7]; };
    const V3 zero{{0.0, 0.0, 0.0}};
    double cfl = 0.0;
    std::vector<V3> S(PX * PY, zero), FM(PX * PY, zero), FP(PX * PY, zero), GM(PX * PY, zero), GP(PX * PY, zero),
        AM(PX * PY, zero), AP(PX * PY, zero), A(PX * PY, zero), B(PX * PY, zero);
    std::vector<V7> E(PX * PY);
    const auto vel = [&](int k) { return fast::cell_velocity(h[k], hu[k], hv[k], g); };
    // one direction's Riemann problems, limiter and corrections (n, t: its momenta)
    const auto faces = [&](int dir, double dtd) {
        const std::vector<double>&n = dir ? hv : hu, &t = dir ? hu : hv;
        double smax = 0.0, c2 = 0.0;
        for (int j = 0; j < PY - (dir ? 0 : 1); j++)
            for (int i = 0; i < PX - (dir ? 1 : 0); i++) {
                const int p = at(i, j), kR = ti(i, j), kL = dir ? ti(i, j - 1) : ti(i - 1, j);
                double s[3] = {0, 0, 0}, w[7] = {0, 0, 0, 0, 0, 0, 0};
                if (fast_form) {
                    fast::CellVel L = vel(kL), R = vel(kR);
                    if (dir) std::swap(L.u, L.v), std::swap(R.u, R.v);
                    fast::rpn2_face(h[kL], n[kL], t[kL], bed[kL], h[kR], n[kR], t[kR], bed[kR], L, R, P, s, w);
                    for (int m = 0; m < 3; m++) smax = fast::vmax(smax, std::fabs(s[m]));
                } else {
                    double w3[3][3];
                    rpn2_face(h[kL], n[kL], t[kL], bed[kL], h[kR], n[kR], t[kR], bed[kR], P, s, w3);
                    compress(w3, w);
                    for (int m = 0; m < 3; m++) {
                        c2 = fmaxf64(c2, dtd * s[m]);
                        c2 = fmaxf64(c2, -(dtd * s[m]));
                    }
                }
                std::memcpy(S[p].v, s, sizeof s);
                std::memcpy(E[p].v, w, sizeof w);
            }
        cfl = fmaxf64(cfl, fast_form ? dtd * smax : c2);
        const int step = dir ? PX : 1;
        for (int j = dir; j <= ny + 1; j++)
            for (int i = 1 - dir; i <= nx + 1; i++) {
                const int p = at(i, j);
                double wn[7], fm[3], fp[3];
                const auto from = [&](int f) { return E[S[p].v[f] > 0.0 ? p - step : p + step].v; };
                for (int k = 0; k < 3; k++) {
                    wn[k] = from(0)[k];
                    wn[4 + k] = from(2)[4 + k];
                }
                wn[3] = from(1)[3];
                if (dir && fast_form) fast::face_second_order<1, false>(E[p].v, S[p].v, wn, dtd, P, fm, fp, AM[p].v, AP[p].v);
                else if (fast_form) fast::face_second_order<0, false>(E[p].v, S[p].v, wn, dtd, P, fm, fp, AM[p].v, AP[p].v);
                else if (dir) face_second_order<1, false>(E[p].v, S[p].v, wn, dtd, P, fm, fp, AM[p].v, AP[p].v);
                else face_second_order<0, false>(E[p].v, S[p].v, wn, dtd, P, fm, fp, AM[p].v, AP[p].v);
                V3&m = dir ? GM[p] : FM[p], &o = dir ? GP[p] : FP[p];
                for (int k = 0; k < 3; k++) {
                    const int l = dir && k ? 3 - k : k;
                    m.v[k] = dir ? m.v[k] + fm[l] : fm[l];
                    o.v[k] = dir ? o.v[k] + fp[l] : fp[l];
                }
            }
    };
    // transverse increments of cell (i, j): A on its low side, B on its high side
    const auto split = [&](int dir, int i, int j, double hd) {
        const int p = at(i, j), k = ti(i, j), next = dir ? p + PX : p + 1;
        const int lo = dir ? ti(i - 1, j) : ti(i, j - 1), hi = dir ? ti(i + 1, j) : ti(i, j + 1);
        if (fast_form) {
            const fast::CellVel c = vel(k);
            fast::cell_transverse(fast::rpt2_setup(h[k], dir ? c.v : c.u, dir ? c.u : c.v, c.sg, bed[k], bed[lo], bed[hi], tol),
                                  AM[next].v, AP[p].v, hd, A[p].v, B[p].v);
        } else {
            cell_transverse(rpt2_setup(h[k], dir ? hv[k] : hu[k], dir ? hu[k] : hv[k], bed[k], bed[lo], bed[hi], g, tol),
                            AM[next].v, AP[p].v, hd, A[p].v, B[p].v);
        }
    };
    if (wet) {
        faces(0, dtdx);
        if (P.transverse)
            for (int j = 0; j <= ny + 1; j++)
                for (int i = 1; i <= nx; i++) split(0, i, j, 0.5 * dtdx);
        for (int j = 1; j <= ny + 1; j++)
            for (int i = 1; i <= nx; i++)
                for (int k = 0; k < 3; k++) GM[at(i, j)].v[k] = GP[at(i, j)].v[k] = B[at(i, j - 1)].v[k] + A[at(i, j)].v[k];
        std::fill(AM.begin(), AM.end(), zero);
        std::fill(AP.begin(), AP.end(), zero);
        std::fill(A.begin(), A.end(), zero);
        std::fill(B.begin(), B.end(), zero);
        faces(1, dtdy);
        if (P.transverse)
            for (int j = 1; j <= ny; j++)
                for (int i = 0; i <= nx + 1; i++) split(1, i, j, 0.5 * dtdy);
        for (int j = 1; j <= ny; j++)
            for (int i = 1; i <= nx + 1; i++)
                for (int k = 0; k < 3; k++) {
                    const int l = k ? 3 - k : k, p = at(i, j);
                    FM[p].v[k] = FM[p].v[k] + B[p - 1].v[l] + A[p].v[l];
                    FP[p].v[k] = FP[p].v[k] + B[p - 1].v[l] + A[p].v[l];
                }
    }
    for (int j = 1; j <= ny; j++)
        for (int i = 1; i <= nx; i++) {
            const int k = ti(i, j), p = at(i, j);
            double v[3] = {h[k], hu[k], hv[k]};
            if (wet)
                for (int m = 0; m < 3; m++)
                    v[m] = v[m] - dtdx * (FM[p + 1].v[m] - FP[p].v[m]) - dtdy * (GM[p + PX].v[m] - GP[p].v[m]);
            if (P.src_term > 0) {
                if (fast_form && wet) fast::src2_cell(v[0], v[1], v[2], bed[k], dt, P);
                else src2_cell(v[0], v[1], v[2], bed[k], dt, P);
            }
            for (int m = 0; m < 3; m++) q[3 * k + m] = v[m];
        }
    return cfl;
}
}  // namespace gf
'''


def _lib():
    global _LIB
    if _LIB is None:
        d = tempfile.mkdtemp(prefix="gf_phys_")
        os.makedirs(os.path.join(d, "hip"))
        open(os.path.join(d, "hip", "hip_runtime.h"), "w").close()
        src = os.path.join(d, "p.cpp")
        with open(src, "w") as f:
            f.write(_SRC)
        so = os.path.join(d, "p.so")
        subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-I", d,
                        "-I", os.path.join(ROOT, "geoflood_amd", "csrc"), "-o", so, src], check=True)
        _LIB = ct.CDLL(so)
        _LIB.gf_host_step.restype = ct.c_double
    return _LIB


def host_step(params, q, bed, dx, dy, dt, fast):
    """One step of a patch (q: (ny+4, nx+4, 3), updated in place) with the fast
    or the general operations.  Returns (largest CFL number, in the range)."""
    dp = ct.POINTER(ct.c_double)
    ok = ct.c_int()
    cp = params.to_c()
    assert q.flags.c_contiguous and bed.flags.c_contiguous and q.shape[:2] == bed.shape[:2]
    cfl = _lib().gf_host_step(int(fast), q.shape[1] - 4, q.shape[0] - 4, q.ctypes.data_as(dp), bed.ctypes.data_as(dp),
                              ct.c_double(dx), ct.c_double(dy), ct.c_double(dt), ct.byref(cp), ct.byref(ok))
    return cfl, bool(ok.value)
