// Boundary-site arithmetic (GridClass::applyBCs, regularisedBC,
// convectiveBC, Grid.cpp:302-474) shared by the boundary kernels: FP64 with
// the reference's operation order, for both storages.
//
// Nine lanes work on one site, lane v on population v: a site's arithmetic
// is several times a bulk collision's and there are only O(Nx + Ny) sites,
// so with one lane per site the whole time is one long dependent chain on a
// few wavefronts.  Split over the populations, a lane evaluates two
// equilibria instead of eighteen and the chain is about a third as long.
// Sums over the populations are formed by every lane, in v order from zero,
// so each value is the one a single lane would compute.
#pragma once

#include "d2q9_f64.h"

namespace life {

constexpr int kBCLanes = kNV;            // lanes per boundary site
constexpr int kBCPerWave = 64 / kBCLanes;  // sites per wavefront (one lane left over)

// feq64 with a run-time lattice velocity (cx, cy: -1, 0 or 1).
template <bool CM>
LIFE_DI double feq64_rt(double rho, double ux, double uy, double cx, double cy, double w) {
    if (CM) {
        double ax = 9.0 * (cx * cx) * (ux * ux) + 6.0 * cx * ux - 3.0 * (ux * ux) + 2.0;
        double ay = 9.0 * (cy * cy) * (uy * uy) + 6.0 * cy * uy - 3.0 * (uy * uy) + 2.0;
        return 0.25 * rho * w * ax * ay;
    } else {
        double cu = cx * ux + cy * uy;
        double q = ux * ux * (cx * cx - 1.0 / 3.0) + uy * uy * (cy * cy - 1.0 / 3.0);
        return rho * w * (1.0 + 3.0 * cu + 4.5 * q + 9.0 * cx * cy * ux * uy);
    }
}

// Orders LDS writes of some lanes before later reads by other lanes of the
// same wavefront.
LIFE_DI void bc_lane_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// What lane v of a boundary site knows before any population is read.
struct BCLane {
    int v, vo;           // its population and the opposite one
    int p[3], z[3];      // populations leaving through the side, and along it, in v order
    int type, nd;
    double nn;           // inward normal along nd
    bool corner, unknown, buried;
    bool nbr;            // the site reads its two inward neighbours: the zero gradient of
                         // free-slip and pressure sites, the density extrapolation of corners
    double cx, cy, w, wq;
};

LIFE_DI BCLane bc_lane(const GridScalars& g, int v, int type, int nx, int ny, int nd) {
    BCLane l;
    l.v = v;
    l.vo = v == 0 ? 0 : ((v - 1) ^ 1) + 1;
    const int cx = v == 1 || v == 5 || v == 7 ? 1 : (v == 2 || v == 6 || v == 8 ? -1 : 0);
    const int cy = v == 3 || v == 5 || v == 8 ? 1 : (v == 4 || v == 6 || v == 7 ? -1 : 0);
    l.type = type;
    l.nd = nd;
    const int nn = nd == 0 ? nx : ny;
    l.nn = nn;
    l.corner = nx != 0 && ny != 0;
    l.nbr = type == 3 || type == 4 || l.corner;
    // populations that entered from outside the domain; at a corner, those
    // along the diagonal between its sides have no opposite to take
    l.unknown = l.corner ? (cx == nx || cy == ny) : (nd == 0 ? cx == nx : cy == ny);
    l.buried = l.corner && nx * cx + ny * cy == 0;
    l.p[0] = nd == 0 ? (nn > 0 ? 2 : 1) : (nn > 0 ? 4 : 3);
    l.p[1] = nn > 0 ? 6 : 5;
    l.p[2] = nd == 0 ? (nn > 0 ? 8 : 7) : (nn > 0 ? 7 : 8);
    l.z[0] = 0;
    l.z[1] = nd == 0 ? 3 : 1;
    l.z[2] = nd == 0 ? 4 : 2;
    l.cx = cx;
    l.cy = cy;
    l.w = w64(v);
    l.wq = v == 0 ? g.wq[0] : (v < 5 ? g.wq[1] : g.wq[2]);
    return l;
}

// Density and the velocity along the side (momentum + F/2 over density,
// moments64) of a neighbour's populations.
LIFE_DI void bc_neighbour(const double f[kNV], int nd, double F, double& r, double& ut) {
    double s = 0.0, m = 0.0;
#pragma unroll
    for (int v = 0; v < kNV; v++) {
        s += f[v];
        m += (nd != 0 ? kCX[v] : kCY[v]) * f[v];
    }
    r = s;
    ut = (m + 0.5 * F) / s;
}

// The site's post-stream populations that lane l reads: those leaving
// through the side, those along it, its own and the opposite one.  get(v, w):
// population v, whose weight is w.
struct BCPops {
    double p[3], z[3], f, fo;
};
template <typename G>
LIFE_DI BCPops bc_read(const BCLane& l, G&& get) {
    BCPops q;
    q.p[0] = get(l.p[0], 1.0 / 9.0);
    q.p[1] = get(l.p[1], 1.0 / 36.0);
    q.p[2] = get(l.p[2], 1.0 / 36.0);
    q.z[0] = get(l.z[0], 4.0 / 9.0);
    q.z[1] = get(l.z[1], 1.0 / 9.0);
    q.z[2] = get(l.z[2], 1.0 / 9.0);
    q.f = get(l.v, l.w);
    q.fo = get(l.vo, l.w);
    return q;
}

// applyBCs + regularisedBC of one wall, velocity, free-slip or pressure site:
// the value of population l.v.  r1, u1, r2, u2: density and velocity along
// the side of the inward neighbours (used only with l.nbr); uwx, uwy: u_in
// times the ramp; rho_in; pun: the site's previous velocity across the side
// (used only at a pressure corner: everywhere else rho_n and u_n of the
// previous step are overwritten); share: kNV entries of LDS of the site's
// own.  All lanes of the site call it together.  Selects, not branches: the
// sites of a wavefront may be of several types.
template <bool CM>
LIFE_DI double bc_value(const BCLane& l, const GridScalars& g, const BCPops& q, double r1, double u1, double r2,
                        double u2, double uwx, double uwy, double rho_in, double pun, double* share) {
    const bool pressure = l.type == 4, inlet = l.type == 2;
    // velocity across and along the side
    double un = inlet ? (l.nd == 0 ? uwx : uwy) : 0.0;
    double ut = inlet ? (l.nd == 0 ? uwy : uwx) : 0.0;
    // Utils::zeroGradient order 2 on the current velocity (Utils.h:200-210)
    const double ext = (4.0 / 3.0) * u1 - (1.0 / 3.0) * u2;
    ut = l.type >= 3 ? ext : ut;
    // regularisedBC, Grid.cpp:400-425: density from the known populations
    // (pressure: the velocity across); a corner extrapolates its density
    // (Utils.h:150-162)
    const double fplus = ((0.0 + q.p[0]) + q.p[1]) + q.p[2], fzero = ((0.0 + q.z[0]) + q.z[1]) + q.z[2];
    const double d = (2.0 * fplus + fzero) / (pressure ? rho_in : 1.0 - l.nn * un);
    double rn = pressure ? rho_in : (l.corner ? 2.0 * r1 - r2 : d);
    un = pressure ? (l.corner ? pun : l.nn * (1.0 - d)) : un;
    const double uxn = l.nd == 0 ? un : ut, uyn = l.nd == 0 ? ut : un;
    const double feq = feq64_rt<CM>(rn, uxn, uyn, l.cx, l.cy, l.w);
    const double feqo = feq64_rt<CM>(rn, uxn, uyn, -l.cx, -l.cy, l.w);
    const double f = l.unknown ? (l.buried ? feq : feq + (q.fo - feqo)) : q.f;
    share[l.v] = f - feq;
    bc_lane_fence();
    double fneq[kNV];
#pragma unroll
    for (int v = 0; v < kNV; v++) fneq[v] = share[v];
    bc_lane_fence();  // share may be rewritten after the call
    // sums of c c f_neq in v order: the terms with c = 0 add nothing (that of
    // the rest population is kept for a NaN there)
    const double s0 = 0.0 * fneq[0];
    const double Sxx = s0 + fneq[1] + fneq[2] + fneq[5] + fneq[6] + fneq[7] + fneq[8];
    const double Syy = s0 + fneq[3] + fneq[4] + fneq[5] + fneq[6] + fneq[7] + fneq[8];
    const double Sxy = s0 + fneq[5] + fneq[6] - fneq[7] - fneq[8];
    return feq + l.wq * (((l.cx * l.cx - g.cs2) * Sxx) + ((l.cy * l.cy - g.cs2) * Syy) + (2.0 * l.cx * l.cy * Sxy));
}

// convectiveBC (Grid.cpp:468-474): the value of population v = 2, 6 or 8 at
// an outlet site from its value fn before the step.
LIFE_DI double bc_convective(int v, double fn, double dux, double duy) {
    return fn + 3.0 * w64(v) * (dux * -1 + duy * (v == 2 ? 0 : (v == 6 ? -1 : 1)));
}

}  // namespace life
